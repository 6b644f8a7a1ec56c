"""The wave-split FP64 and chunked matrix-core shallow-water sums at the edges
of their shapes (sources around a quad and the chunk rule's steps, targets around a block of
64), against the oracle, and the form without a partial-sum workspace, which
must give the same bits.

Tolerance: targets are vertices and sources leaf faces of the icosahedral
mesh of level 3, so 1 - x.y >= 1.5e-3 and its rounding of 1.1e-16 changes a
pair's 1 / (1 - x.y) by at most 8e-14 and the double dot, quadratic in sums of
its squares, by four times that, 3e-13.
"""
import numpy as np
import pytest

from conftest import aos, mesh

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from lpm_amd import _abi  # noqa: E402

TOL = 1e-12


@pytest.fixture(scope="module")
def ctx():
    from lpm_amd.device import Context
    c = Context(0)
    yield c
    c.close()


def dev(a, dtype=torch.float64):
    return torch.tensor(np.ascontiguousarray(a), dtype=dtype, device="cuda")


def _inputs(ns, depth=3):
    m = mesh(0, depth)
    x = m.face_x[:, m.leaf_slice][:, :ns]
    area = m.face_area[m.leaf_slice][:ns]
    surf = lambda p: 1 + 0.3 * np.cos(2 * p[0]) + 0.1 * p[2]  # noqa: E731
    return (m, x, area, np.sin(3 * x[0]) + x[2], 0.3 * np.cos(2 * x[1]), surf)


def _close(got, ref):
    assert np.linalg.norm(got - ref) <= TOL * np.linalg.norm(ref)


@pytest.mark.parametrize("ns", [1, 4, 5, 159, 161, 319, 321, 1280])
@pytest.mark.parametrize("nt", [1, 63, 64, 65, 129, 642])
@pytest.mark.parametrize("eps", [0.0, 0.1])
def test_free_targets_match_oracle(ctx, ora, ns, nt, eps):
    m, x, area, zeta, sigma, surf = _inputs(ns)
    t = m.vert_x[:, :nt]
    got = ctx.swe_sums(dev(t), dev(surf(t)), dev(x), dev(zeta), dev(sigma),
                       dev(area), dev(surf(x)), eps=eps, pse_eps=0.3)
    ref = ora.swe_sums(aos(t), surf(t), aos(x), zeta, sigma, area, surf(x),
                       np.zeros(ns, np.uint8), eps=eps, pse_eps=0.3)
    for g, r in zip(got, ref):
        _close(g.cpu().numpy().T, r)


@pytest.mark.parametrize("pse_eps", [0.05, 0.13, 0.15])
@pytest.mark.parametrize("r", [1.0, 0.5])
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_pse_terms_match_oracle(ctx, ora, pse_eps, r, prec):
    # cut-off radii (7.07 pse_eps) on both sides of |x|, the bound that implies
    # x.y > 0.  exp(-z) is off by z times the rounding of rho^2, at most
    # 50 * 4 * 1.1e-16, and its own 2 units: 2.3e-14 of a term.  The terms left
    # out are below exp(-50) of theirs.
    m, x, area, zeta, sigma, surf = _inputs(1280)
    t = r * m.vert_x
    got = ctx.swe_sums(dev(t), dev(surf(t)), dev(x), dev(zeta), dev(sigma),
                       dev(area), dev(surf(x)), eps=0.1, pse_eps=pse_eps,
                       precision=prec)[2]
    ref = ora.swe_sums(aos(t), surf(t), aos(x), zeta, sigma, area, surf(x),
                       np.zeros(1280, np.uint8), eps=0.1, pse_eps=pse_eps)[2]
    cut = (np.exp(-50) * 4 / (np.pi * pse_eps ** 4) *
           (area * np.abs(surf(x) - surf(t)[:, None])).sum(1))
    assert (np.linalg.norm(got.cpu().numpy() - ref) <=
            TOL * np.linalg.norm(ref) + np.linalg.norm(cut))


@pytest.mark.parametrize("ns", [2, 65, 161, 1280])
def test_collocated_targets_match_oracle(ctx, ora, ns):
    m, x, area, zeta, sigma, surf = _inputs(ns)
    mask = np.zeros(ns, np.uint8)
    mask[1::5] = 1
    for flags in (0, _abi.LPM_FLAG_SKIP_MASKED_TARGETS):
        got = ctx.swe_sums(dev(x), dev(surf(x)), dev(x), dev(zeta), dev(sigma),
                           dev(area), dev(surf(x)), dev(mask, torch.uint8),
                           collocated=True, eps=0.0, pse_eps=0.3, flags=flags)
        ref = ora.swe_sums(aos(x), surf(x), aos(x), zeta, sigma, area, surf(x),
                           mask, collocated=True, eps=0.0, pse_eps=0.3)
        live = (mask == 0) | (flags == 0)
        for g, r in zip(got, ref):
            _close(g.cpu().numpy().T[live], r[live])


@pytest.mark.parametrize("ns", [1, 255, 257, 1366, 5119])
@pytest.mark.parametrize("nt", [1, 63, 65, 257, 2562])
def test_mixed_matches_fp64(ctx, ns, nt):
    # 1e-6: the bound of the mixed sums (FP32 far field, 22-bit operands)
    m, x, area, zeta, sigma, surf = _inputs(ns, 4)
    t = m.vert_x[:, :nt]
    arg = (dev(t), dev(surf(t)), dev(x), dev(zeta), dev(sigma), dev(area),
           dev(surf(x)))
    a = ctx.swe_sums(*arg, eps=0.05, pse_eps=0.3, precision="mixed")
    b = ctx.swe_sums(*arg, eps=0.05, pse_eps=0.3)
    for g, r in zip(a, b):
        assert torch.linalg.norm(g - r) <= 1e-6 * torch.linalg.norm(r)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_without_a_workspace_the_bits_are_the_same(prec):
    """Captured by the caller in a context whose partial-sum workspace is too
    small, each block sums every chunk itself."""
    from lpm_amd.device import Context
    c = Context(0)
    try:
        m, x, area, zeta, sigma, surf = _inputs(5120, 4)
        t = m.vert_x[:, :500]
        src = [dev(a) for a in (x, zeta, sigma, area, surf(x))]
        tx, ts = dev(t), dev(surf(t))
        kw = dict(eps=0.05, pse_eps=0.1, precision=prec)
        # sizes the packed sources, and what 500 targets need without chunks
        c.swe_sums(tx[:, :1], ts[:1], *src, **kw)
        c.swe_sums(tx, ts, src[0][:, :256], *(a[:256] for a in src[1:]), **kw)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.graph(g, stream=side):
            got = c.swe_sums(tx, ts, *src, **kw)
        want = c.swe_sums(tx, ts, *src, **kw)
        for _ in range(3):
            for a in got:
                a.zero_()
            g.replay()
            torch.cuda.synchronize()
            for a, b in zip(got, want):
                assert torch.equal(a, b)
        del g
    finally:
        c.close()


@pytest.mark.parametrize("ns", [1, 5, 127, 128, 129])
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_many_targets_over_few_sources(ctx, ora, ns, prec):
    """From 32,768 arbitrary targets on, 128 sources or fewer are summed by one
    wave for all of them, in FP64 also where mixed precision is asked for."""
    m, x, area, zeta, sigma, surf = _inputs(ns, 4)
    t = np.tile(m.vert_x, 13)[:, :32769]
    src = [dev(a) for a in (x, zeta, sigma, area, surf(x))]
    kw = dict(eps=0.05, pse_eps=0.3, precision=prec)
    ref = ora.swe_sums(aos(t[:, :2562]), surf(t[:, :2562]), aos(x), zeta, sigma,
                       area, surf(x), np.zeros(ns, np.uint8), eps=0.05,
                       pse_eps=0.3)
    for n in (32767, 32768, 32769):
        got = ctx.swe_sums(dev(t[:, :n]), dev(surf(t[:, :n])), *src, **kw)
        for g, r in zip(got, ref):
            g = g.cpu().numpy()
            # (the matrix-core passes' near tiles depend on a wave's targets)
            few = prec == "fp64" or (n >= 32768 and ns <= 128)
            if few:
                assert np.array_equal(g[..., 2562:5124], g[..., :2562])
            assert (np.linalg.norm(g[..., :2562].T - r) <=
                    (TOL if few else 1e-6) * np.linalg.norm(r))
