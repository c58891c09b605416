"""Single-direction column strips and the element-wise sweeps against numpy in 64 bits.

Tolerances: a 2-D transform is 2*log2(n) rounded butterfly levels of rms relative error
about 2^-24 (2^-53), adding in quadrature: 2.9e-7 at 4096 points, doubled for twiddles and
factors; an element-wise product is 2 roundings plus the factor's 3: 2^-24 * 5.
"""
import numpy as np
import pytest
import torch

from conftest import rel_l2
import oracle
from oracle.angular_spectrum import construct_grids

pytestmark = pytest.mark.gpu
DEV = "cuda"
AREA, WL, Z = 400e-4, 632e-7, 50e-4
TOL = {"c64": 5.9e-7, "c128": 1.1e-15}
TOL_E = {"c64": 3.0e-7, "c128": 1e-9}  # 64 bits: the phase Kz*z itself, 1e5 turns of 1e-15


def _rand(shape, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(shape, dtype=torch.complex64 if dtype == "c64" else torch.complex128,
                       generator=g)


def _factor(n, ap):
    g = construct_grids(AREA, n, WL)
    h = oracle.transfer_function(g.Kz, Z)
    f = np.fft.fftfreq(n, AREA / n)
    return h * (f[None, :] ** 2 + f[:, None] ** 2 <= ap * ap)


@pytest.mark.parametrize("n,batch,dtype", [
    (128, 3, "c128"), (256, 2, "c64"), (256, 3, "c128"), (512, 2, "c64"), (512, 1, "c128"),
    (1024, 1, "c64"), (1024, 5, "c64"), (1024, 2, "c128"), (2048, 1, "c64"), (2048, 1, "c128"),
    (4096, 1, "c64"), (4096, 1, "c128")])
def test_single_direction_passes(n, batch, dtype):
    from lightprop2d_amd import propagation as P
    u = _rand((batch, n, n), dtype, n)
    w = u.numpy().astype(np.complex128)
    spec = np.fft.fft2(w)
    assert rel_l2(P.fft2(u.to(DEV)).cpu().numpy(), spec) < TOL[dtype]
    assert rel_l2(P.ifft2(u.to(DEV)).cpu().numpy(), np.fft.ifft2(w)) < TOL[dtype]
    # spectral stage with a pupil, then the inverse transform; what lies outside the pupil
    # (an infinity here) leaves no trace
    ap = 0.4 * n / AREA
    f = _factor(n, ap)
    s, field = u.to(DEV), torch.empty_like(u, device=DEV)
    outside = np.argwhere(f == 0)
    y, x = outside[len(outside) // 2]
    s[:, y, x] = float("inf")
    w[:, y, x] = 0
    P.spectral_apply(s, z=Z, area_size=AREA, wl=WL, aperture_radius=ap, field_out=field)
    tol = TOL[dtype] if dtype == "c64" else TOL_E[dtype]
    assert rel_l2(field.cpu().numpy(), np.fft.ifft2(w * f)) < tol
    assert torch.all(s[:, y, x] == 0)


@pytest.mark.parametrize("dtype", ["c64", "c128"])
@pytest.mark.parametrize("n,batch", [(2, 5), (4, 1), (16, 4097), (256, 3), (1024, 1)])
def test_elementwise_sweeps_at_any_alignment(n, batch, dtype):
    """16-byte aligned planes and planes one element further on."""
    from lightprop2d_amd import propagation as P
    u = _rand((batch * n * n + 1,), dtype, n + batch)
    f = _factor(n, 0.4 * n / AREA)
    mask = np.random.RandomState(n).uniform(0.5, 1.5, (n, n)).astype(np.float32)
    for off in (0, 1):
        w = u[off:off + batch * n * n].reshape(batch, n, n).numpy().astype(np.complex128)
        for m in ((), (mask,), (mask, mask)):
            buf = u.to(DEV)
            v = buf[off:off + batch * n * n].view(batch, n, n)
            P.spectral_apply(v, masks=[torch.from_numpy(q).to(DEV) for q in m], z=Z,
                             area_size=AREA, wl=WL, aperture_radius=0.4 * n / AREA)
            exp = w * f
            for q in m:
                exp = exp * q
            assert rel_l2(v.cpu().numpy(), exp) < TOL_E[dtype], (off, len(m))
        buf = u.to(DEV)
        v = buf[off:off + batch * n * n].view(batch, n, n)
        got = P.intensity(v).cpu().numpy()
        exp = w.real.astype(np.longdouble) ** 2 + w.imag.astype(np.longdouble) ** 2
        assert np.abs(got - exp).max() <= 2.0 ** (-22 if dtype == "c64" else -51) * exp.max()
        P.spatial_apply(v, masks=[torch.from_numpy(mask).to(DEV)])
        assert rel_l2(v.cpu().numpy(), w * mask) < TOL_E[dtype]


@pytest.mark.parametrize("shape,batch", [((1,), 1), ((5, 5), 3), ((17,), 4097), ((32, 32), 64),
                                         ((33, 31), 300), ((128, 128), 65), ((512, 512), 4),
                                         ((1024, 1024), 3)])
def test_sum_of_planes(shape, batch):
    """Every number of slices, odd counts, and the sum written over plane 0.  Whole numbers
    whose sums stay below 2^24: exact in any order."""
    from lightprop2d_amd import propagation as P
    x = torch.randint(-1000, 1001, (batch, *shape), generator=torch.Generator().manual_seed(batch))
    exp = x.sum(0).float()
    x = x.float()
    assert torch.equal(P.sum_planes(x.to(DEV), torch.empty(shape, device=DEV)).cpu(), exp)
    buf = x.to(DEV)
    P.sum_planes(buf, buf[0])
    assert torch.equal(buf[0].cpu(), exp)


@pytest.mark.parametrize("n,n_out", [(1, 3), (2, 4), (3, 5), (4, 6), (510, 514), (512, 1026),
                                     (500, 1024), (1000, 1502), (1024, 1024), (1024, 2050)])
@pytest.mark.parametrize("dtype", ["c64", "c128"])
def test_expand_is_edge_padding(n, n_out, dtype):
    """Even and odd sizes, partial last workgroups of a row, three fields: exact copies."""
    from lightprop2d_amd import propagation as P
    u = _rand((3, n, n), dtype, n)
    d = (n_out - n) // 2
    exp = np.pad(u.numpy(), ((0, 0), (d, d), (d, d)), mode="edge")
    assert np.array_equal(P.expand(u.to(DEV), n_out).cpu().numpy(), exp)
