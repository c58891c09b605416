"""Batches that run in parts, and the column schedules chosen by the size of a part.

A batch whose planes exceed the cache between the sweeps runs chunk by chunk, and at
1024 points a chunk of fewer than four fields takes narrower column strips than a larger
one.  Tolerance: a whole propagation is 4*log2(n) rounded butterfly levels of rms
relative error about 2^-24 each, adding in quadrature: sqrt(4*12)*6e-8 = 4.1e-7 at 4096
points (complex128 8e-16), doubled for the twiddles and the transfer function.
"""
import numpy as np
import pytest
import torch

from conftest import rel_l2
import oracle

pytestmark = pytest.mark.gpu
DEV = "cuda"
AREA, WL, Z = 400e-4, 632e-7, 50e-4
TOL = {"c64": 8.3e-7, "c128": 1.6e-15}


@pytest.fixture
def lib():
    from lightprop2d_amd import propagation as P
    handle = P._lib()
    saved = {(d, n): handle.lp2d_get_chunk(n, d) for d in (0, 1)
             for n in (256, 512, 1024, 2048, 4096)}
    yield handle
    for (d, n), c in saved.items():
        handle.lp2d_set_chunk(n, d, c)


def _field(shape, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(shape, dtype=torch.complex64 if dtype == "c64" else torch.complex128,
                       generator=g)


# (points, fields, fields per chunk): whole and partial last chunks; 1024 points on both
# sides of four fields per chunk
SPLITS = [(256, 5, 2, "c64"), (512, 3, 1, "c64"), (1024, 4, 0, "c64"), (1024, 3, 0, "c64"),
          (1024, 7, 4, "c64"), (2048, 3, 2, "c64"), (4096, 2, 1, "c64"), (256, 5, 2, "c128"),
          (1024, 3, 2, "c128")]


@pytest.mark.parametrize("in_place", [False, True], ids=["out", "in_place"])
@pytest.mark.parametrize("n,batch,chunk,dtype", SPLITS)
def test_split_batch_matches_oracle(lib, n, batch, chunk, dtype, in_place):
    from lightprop2d_amd import propagation as P
    u = _field((batch, n, n), dtype, n + batch)
    scr = torch.rand((batch, n, n), generator=torch.Generator().manual_seed(n)) * 6
    assert lib.lp2d_set_chunk(n, 0 if dtype == "c64" else 1, chunk) == 0
    x = u.to(DEV)
    out = P.propagate(x, Z, AREA, WL, phase=scr.to(DEV), aperture_radius=0.2 / WL,
                      out=x if in_place else None)
    for b in {0, batch - 1}:
        exp = oracle.propagate_field(u[b].numpy(), AREA, WL, Z, aperture_radius=0.2 / WL,
                                     phase_mask=scr[b].numpy().astype(np.float64))
        assert rel_l2(out[b].cpu().numpy(), exp) < TOL[dtype], b


def test_default_split_equals_one_chunk(lib):
    """513 fields of 256 points (one more than the cache holds) and 7 stacked fields:
    the same bits however the batch is split, spectrum output and screens included."""
    from lightprop2d_amd import propagation as P
    u = _field((513, 256, 256), "c64", 1).to(DEV)
    scr = torch.rand((513, 256, 256), device=DEV) * 6
    spec = [torch.empty_like(u) for _ in range(2)]
    got = []
    for k, chunk in enumerate((0, 513)):
        assert lib.lp2d_set_chunk(256, 0, chunk) == 0
        got.append(P.propagate(u, Z, AREA, WL, phase=scr, spectrum_out=spec[k]))
    assert torch.equal(got[0], got[1]) and torch.equal(spec[0], spec[1])
    scr = torch.rand((3, 512, 512), device=DEV) * 6
    u = _field((7, 512, 512), "c64", 2).to(DEV)
    got = []
    for chunk in (0, 2):
        assert lib.lp2d_set_chunk(512, 0, chunk) == 0
        planes = [None] + [torch.empty_like(u) for _ in range(2)]
        got.append([P.propagate_stack(u, scr, Z, AREA, WL, planes=planes), *planes[1:]])
    assert all(torch.equal(a, b) for a, b in zip(*got))


@pytest.mark.parametrize("K", [1, 2, 5])
@pytest.mark.parametrize("n", [256, 1024, 2048, 4096])
def test_stack_and_its_adjoint_match_the_planes(lib, n, K):
    """The chained sweeps and their adjoint (2048 points included) against plane by plane
    calls of propagate and propagate_adjoint; the two are 4*K*log2(n) levels apart."""
    from lightprop2d_amd import propagation as P
    u = _field((2, n, n), "c64", n + K).to(DEV)
    g = _field((2, n, n), "c64", n + K + 1).to(DEV)
    scr = torch.rand((K, n, n), device=DEV) * 6
    tol = 8.3e-7 * (2 * K) ** 0.5
    planes = [u]
    for k in range(K):
        planes.append(P.propagate(planes[-1], Z, AREA, WL, phase=scr[k]))
    out = P.propagate_stack(u, scr, Z, AREA, WL)
    assert rel_l2(out.cpu().numpy(), planes[-1].cpu().numpy()) < tol
    gf, gs = P.propagate_stack_adjoint(g, planes[:-1], scr, Z, AREA, WL)
    x, exp = g, [None] * K
    for k in reversed(range(K)):
        x, exp[k] = P.propagate_adjoint(x, planes[k], Z, AREA, WL, phase=scr[k])
    assert rel_l2(gf.cpu().numpy(), x.cpu().numpy()) < tol
    for k in range(K):
        assert rel_l2(gs[k].cpu().numpy(), exp[k].cpu().numpy()) < tol, k


@pytest.mark.parametrize("n,batch,dtype", [(32, 1, "c64"), (64, 5, "c64"), (128, 2, "c64"),
                                           (128, 300, "c64"), (32, 3, "c128"), (64, 2, "c128"),
                                           (64, 1100, "c128")])
@pytest.mark.parametrize("shared", [True, False], ids=["shared", "per_field"])
def test_whole_field_kernel_with_a_screen(n, batch, dtype, shared):
    """One field per workgroup and several (300 and 1100 fields): forward with a phase
    screen and a pupil, and the adjoint with its phase gradient."""
    from lightprop2d_amd import propagation as P
    ap = 0.4 * n / AREA
    u, g = _field((batch, n, n), dtype, n), _field((batch, n, n), dtype, n + 1)
    ph = torch.rand((n, n) if shared else (batch, n, n),
                    generator=torch.Generator().manual_seed(n + batch)) * 6
    pick = sorted({0, batch // 2, batch - 1})
    out = P.propagate(u.to(DEV), Z, AREA, WL, phase=ph.to(DEV), aperture_radius=ap)
    gin, gph = P.propagate_adjoint(g.to(DEV), u.to(DEV), Z, AREA, WL, phase=ph.to(DEV),
                                   aperture_radius=ap)
    total = np.zeros((n, n))
    for b in range(batch) if shared else pick:
        q = (ph if shared else ph[b]).numpy().astype(np.float64)
        w = np.exp(-1j * q) * oracle.propagate_field(g[b].numpy(), AREA, WL, -Z,
                                                     aperture_radius=ap)
        grad = (np.conj(u[b].numpy().astype(np.complex128)) * w).imag
        total += grad
        if b in pick:
            exp = oracle.propagate_field(u[b].numpy(), AREA, WL, Z, phase_mask=q,
                                         aperture_radius=ap)
            assert rel_l2(out[b].cpu().numpy(), exp) < TOL[dtype], b
            assert rel_l2(gin[b].cpu().numpy(), w) < TOL[dtype], b
            if not shared:
                assert rel_l2(gph[b].cpu().numpy(), grad) < TOL["c64"], b
    if shared:
        assert rel_l2(gph.cpu().numpy(), total) < TOL["c64"]


@pytest.mark.parametrize("n,batch", [(256, 2), (256, 9), (512, 5), (1024, 3), (2048, 2), (4096, 2)])
@pytest.mark.parametrize("lens", [0.0, 0.5])
@pytest.mark.parametrize("field_grad", [True, False])
def test_shared_screen_gradient(lib, n, batch, lens, field_grad):
    """The adjoint of a batch under one screen, with and without a lens and the field's
    gradient, against the per-field screens' path (which sums nothing in the pass)."""
    from lightprop2d_amd import propagation as P
    u, g = _field((batch, n, n), "c64", n).to(DEV), _field((batch, n, n), "c64", n + 1).to(DEV)
    ph = torch.rand((n, n), generator=torch.Generator().manual_seed(n + batch)).to(DEV) * 6
    gin, gph = P.propagate_adjoint(g, u, Z, AREA, WL, phase=ph, lens_f=lens,
                                   aperture_radius=0.2 / WL, want_field_grad=field_grad)
    per = ph.expand(batch, n, n).contiguous()
    exp, parts = P.propagate_adjoint(g, u, Z, AREA, WL, phase=per, lens_f=lens,
                                     aperture_radius=0.2 / WL)
    assert rel_l2(gph.cpu().numpy(), parts.double().sum(0).cpu().numpy()) < 2 * TOL["c64"]
    if field_grad:
        assert rel_l2(gin.cpu().numpy(), exp.cpu().numpy()) < 2 * TOL["c64"]
