"""pyrh_amd.autograd.stokes: the synthesis as a torch.autograd.Function whose
backward is the library's adjoint.  Checked against the response functions
of the same engine, and against central differences of a scalar loss of the
plain FP64 synthesis."""
import numpy as np
import pytest

from pyrh_amd import model, workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng(setups):
    from pyrh_amd.engine import Engine
    e = Engine(model.build_model(setups["lte"], W.wavelengths_630()))
    yield e
    e.close()


@pytest.mark.parametrize("precision", (0, 1))
def test_autograd_backward_is_the_adjoint(eng, precision):
    import torch
    from pyrh_amd import autograd
    from pyrh_amd.engine import RF_PARAMS, RF_ROWS
    atm = W.stokes_map(24, seed=W.SEED_BASE + 81)
    x = torch.from_numpy(atm).cuda().requires_grad_(True)
    st = autograd.stokes(eng, x, mu=1.0, precision=precision)
    ref = eng.synth_lte(atm, precision=precision)
    # the forward runs the adjoint's sweep, which synthesises the same Stokes
    np.testing.assert_allclose(st.detach().cpu().numpy(), ref, rtol=1e-12, atol=0)
    w = torch.linspace(-1.0, 1.0, st.numel(), dtype=torch.float64, device="cuda").view_as(st)
    (st * w).sum().backward()
    g = x.grad.cpu().numpy()
    _, rf = eng.rf_lte(atm, precision=precision)           # [ncol, 6, nd, 4, nout]
    wn = w.cpu().numpy()
    expect = np.einsum("csl,cpksl->cpk", wn, rf.astype(np.float64))
    for ip, row in enumerate(RF_ROWS):
        scale = np.max(np.abs(expect[:, ip]))
        err = np.max(np.abs(g[:, row] - expect[:, ip])) / scale
        print(f"precision {precision} {RF_PARAMS[ip]}: max err {err:.2e}", flush=True)
        assert err < 1e-10
    for row in (0, 2, 8):
        assert np.all(g[:, row] == 0.0)


def test_autograd_against_finite_differences(eng):
    """d L / d T(k) for L = sum of I and d L / d B(k) for L = sum of |V|
    (weights sign(V), held fixed) against central differences of the FP64
    synthesis at depths of the line-forming region, relative to the largest
    gradient of the row.  Weights without cancellation keep the finite
    difference meaningful: the synthesis has kinks (Fritsch-Butland limiter,
    control-point clamps) and Humlicek region boundaries."""
    import torch
    from pyrh_amd import autograd
    atm = W.stokes_map(4, seed=W.SEED_BASE + 82)
    base = eng.synth_lte(atm)
    for row, h, wn in ((1, 0.01, np.zeros_like(base)), (5, 0.1, np.zeros_like(base))):
        if row == 1:
            wn[:, 0] = 1.0
        else:
            wn[:, 3] = np.sign(base[:, 3])
        x = torch.from_numpy(atm).cuda().requires_grad_(True)
        st = autograd.stokes(eng, x, precision=0)
        (st * torch.from_numpy(wn).cuda()).sum().backward()
        g = x.grad.cpu().numpy()
        loss = lambda a: float(np.sum(wn * eng.synth_lte(a)))
        gmax = float(np.max(np.abs(g[:, row].sum(axis=0))))
        for k in (45, 55, 62):
            p, m = atm.copy(), atm.copy()
            p[:, row, k] += h
            m[:, row, k] -= h
            fd = (loss(p) - loss(m)) / (2 * h)
            ad = float(np.sum(g[:, row, k]))
            print(f"row {row} depth {k}: adjoint {ad:.6e}  fd {fd:.6e}  "
                  f"diff/max {abs(ad - fd) / gmax:.2e}", flush=True)
            assert abs(ad - fd) <= 1e-3 * gmax


@pytest.mark.parametrize("ncol,nd,params", [(1, 82, ("T",)), (33, 51, ("B", "T", "vmic")),
                                            (64, 82, ("chi", "gamma")), (97, 37, None)])
@pytest.mark.parametrize("precision", (0, 1))
def test_autograd_contraction_forms(eng, ncol, nd, params, precision):
    """The contraction kernel against torch's, over column and depth counts off
    its tiles, parameter subsets, and gradients that are expanded, transposed
    or float; with create_graph the backward stays differentiable.  The sums
    run over 448 terms in FP64 in another order: 1e-12 of the largest."""
    import torch
    from pyrh_amd import autograd
    from pyrh_amd.engine import RF_PARAMS
    params = params or RF_PARAMS
    atm, _ = W.mixed_batch(ncol, seed=W.SEED_BASE + 83, ndep_choices=(nd,))
    x = torch.from_numpy(atm).cuda().requires_grad_(True)
    st = autograd.stokes(eng, x, precision=precision, params=params)
    g = torch.Generator(device="cuda").manual_seed(3)
    dense = torch.randn(st.shape, generator=g, dtype=torch.float64, device="cuda")
    turned = torch.randn(st.shape[::-1], generator=g, dtype=torch.float64, device="cuda").permute(2, 1, 0)
    one = torch.ones((), dtype=torch.float64, device="cuda").expand(st.shape)
    for grad in (dense, turned, one, dense.float()):
        (a,) = torch.autograd.grad(st, x, grad, retain_graph=True)
        w = grad.clone().requires_grad_(True)
        (b,) = torch.autograd.grad(st, x, w, retain_graph=True, create_graph=True)
        assert b.requires_grad and not a.requires_grad
        c = b.detach()
        assert float((a - c).abs().max()) <= 1e-12 * float(c.abs().max())
        (d,) = torch.autograd.grad(b.sum(), w)      # the Jacobian summed over the rows
        assert d.shape == st.shape and bool(torch.isfinite(d).all()) and float(d.abs().max()) > 0


def _small_graph(eng, ncol=3, precision=0):
    import torch
    from pyrh_amd import autograd
    x = torch.from_numpy(W.stokes_map(ncol, seed=W.SEED_BASE + 84)).cuda().requires_grad_(True)
    st = autograd.stokes(eng, x, precision=precision, params=("T", "B"))
    w = torch.linspace(-1.0, 1.0, 2 * st.numel(), dtype=torch.float64, device="cuda").view(2, *st.shape)
    return x, st, w


@pytest.mark.parametrize("precision", (0, 1))
def test_autograd_carries_forward_tangents(eng, precision):
    """The backward is linear in the incoming gradient, so under forward-mode
    the tangent of a dual gradient goes through the same contraction: to the
    gradient of the tangent (sums in another order, 1e-12 of the largest)."""
    import torch
    import torch.autograd.forward_ad as fad
    x, st, (w, t) = _small_graph(eng, precision=precision)
    (gw,) = torch.autograd.grad(st, x, w, retain_graph=True)
    (gt,) = torch.autograd.grad(st, x, t, retain_graph=True)
    with fad.dual_level():
        (g,) = torch.autograd.grad(st, x, fad.make_dual(w, t), retain_graph=True)
        primal, tangent = fad.unpack_dual(g)
        assert tangent is not None
        for a, b in ((primal, gw), (tangent, gt)):
            assert float((a - b).abs().max()) <= 1e-12 * float(b.abs().max())


def test_autograd_backward_can_be_traced(eng):
    """make_fx records the backward's operations: the graph replays the
    gradient of other incoming gradients too."""
    import torch
    from torch.fx.experimental.proxy_tensor import make_fx
    x, st, (w, t) = _small_graph(eng)
    backward = lambda g: torch.autograd.grad(st, x, g, retain_graph=True)[0]
    graph = make_fx(backward)(w)
    for g in (w, t):
        a, b = graph(g), backward(g)
        assert float((a - b).abs().max()) <= 1e-12 * float(b.abs().max())
