"""A cluster member that gives up waiting is reported, and its call's outputs are NaN,
or are made by the kernels behind the clusters where those are an addition to a
plan that never waited.

The failure is forced from the host: a wait budget of 0 ticks makes every
member leave at its first exchange (ltc_set_cluster_spin_ticks), so every
kernel still exits normally. The call then overwrites every output it writes
with NaN and raises the device's fault flag, which ltc_device_status()
reports and clears.
"""

from __future__ import annotations

import contextlib

import pytest
import torch

import ltc_cuda
from _gpu_common import DEV, _native, _perturbed_module, boundary, gpu_backward, gpu_forward  # noqa: F401

pytestmark = pytest.mark.gpu

T, D, H = 2, 8, 256
DEFAULT_TICKS = 20000000
# Batch sizes at H = 256: one row per cluster in the forward and the chain
# (the one-group kernels), one-row forward and two-row chain clusters, and
# four-row forward and eight-row chain clusters (the two-group kernels).
BATCHES = [16, 48, 200]


@pytest.fixture(params=BATCHES, ids=lambda b: f"B{b}")
def B(request):
    return request.param


@pytest.fixture()
def capi(B):
    c = ltc_cuda._cuda_module.capi
    plan = c.plan(B, T, D, H, 6)
    assert plan["CP"] > 0
    print(f"B={B}: forward rows per cluster {plan['NB']}, chain {plan['NBB']}", flush=True)
    c.device_status(clear=True)  # start clean
    yield c
    assert c.lib.ltc_set_cluster_spin_ticks(DEFAULT_TICKS) >= 0
    c.lib.ltc_device_status(1)


@pytest.fixture()
def capi_row():
    """The library, for the single-workgroup give-up tests (no cluster plan)."""
    c = ltc_cuda._cuda_module.capi
    c.device_status(clear=True)
    yield c
    assert c.lib.ltc_set_cluster_spin_ticks(DEFAULT_TICKS) >= 0
    c.lib.ltc_device_status(1)


class _NoWait:
    """Wait budget of 0 ticks inside the block, the default after it."""

    def __init__(self, capi):
        self.capi = capi

    def __enter__(self):
        assert self.capi.lib.ltc_set_cluster_spin_ticks(0) == DEFAULT_TICKS

    def __exit__(self, *exc):
        assert self.capi.lib.ltc_set_cluster_spin_ticks(DEFAULT_TICKS) == 0


def _expect_fault(capi):
    rc = capi.lib.ltc_device_status(1)
    assert rc == 3 and "gave up" in capi.last_error(), (rc, capi.last_error())
    assert capi.lib.ltc_device_status(0) == 0  # the first read cleared it


def test_forward_give_up_sets_every_output_to_nan(capi, B):
    args = boundary(B, T, D, H, seed=31)
    with _NoWait(capi):
        _, (out, h, saved) = gpu_forward(args, save=True)
    assert torch.isnan(out).all() and torch.isnan(h).all() and torch.isnan(saved).all()
    _expect_fault(capi)
    # the default budget again: finite results and a clean status
    _, (out, h, saved) = gpu_forward(args, save=True)
    assert torch.isfinite(out).all() and torch.isfinite(h).all()
    capi.device_status()


def test_backward_give_up_sets_every_gradient_to_nan(capi, B):
    args = boundary(B, T, D, H, seed=32)
    dev_args, (out, h, saved) = gpu_forward(args, save=True)
    assert torch.isfinite(out).all()
    g_out = torch.randn(B, T, H, device=DEV)
    g_h = torch.randn(B, H, device=DEV)
    with _NoWait(capi):
        grads = gpu_backward(dev_args, saved, g_out, g_h)
    for g in grads:
        assert torch.isnan(g).all()
    _expect_fault(capi)
    grads = gpu_backward(dev_args, saved, g_out, g_h)
    for g in grads:
        assert torch.isfinite(g).all()
    capi.device_status()


def test_module_path_give_up_is_reported_through_python(capi, B):
    m = _perturbed_module(D, H, seed=33).to(DEV)
    x = torch.randn(B, T, D, device=DEV)
    with _NoWait(capi):
        out, (h, _) = m(x)
        out.sum().backward()
    assert torch.isnan(out).all() and torch.isnan(h).all()
    for n, p in m.named_parameters():
        assert torch.isnan(p.grad).all(), n
    with pytest.raises(RuntimeError, match="gave up"):
        ltc_cuda.device_status()
    ltc_cuda.device_status()  # cleared by the call that raised


@pytest.mark.parametrize("D1", [128, 48])
def test_fused_row_backward_give_up_sets_every_gradient_to_nan(capi_row, D1):
    capi = capi_row
    """At H = 64 the module backward's sensory and LayerNorm part runs in
    companion workgroups that wait for the chain's words: with a budget of 0
    they leave at once, and the finalize writes NaN into every gradient."""
    B1, T1, H1 = 24, 8, 64
    plan = capi.plan(B1, T1, D1, H1, 6)
    assert plan["CP"] == 0 and plan["Hp"] == 64 and plan["NB"] == 1 and plan["fuse"] == 1, plan
    m = _perturbed_module(D1, H1, seed=34).to(DEV)
    x = torch.randn(B1, T1, D1, device=DEV, requires_grad=True)
    h0 = (torch.randn(B1, H1, device=DEV) * 0.2).requires_grad_(True)
    out, (h, _) = m(x, (h0, h0))
    assert torch.isfinite(out).all()
    with _NoWait(capi):
        (out.sum() + h.sum()).backward()
    assert torch.isnan(x.grad).all() and torch.isnan(h0.grad).all()
    for n, p in m.named_parameters():
        assert torch.isnan(p.grad).all(), n
    _expect_fault(capi)
    m.zero_grad(set_to_none=True)
    x.grad = h0.grad = None
    out, (h, _) = m(x, (h0, h0))
    (out.sum() + h.sum()).backward()
    assert torch.isfinite(x.grad).all() and torch.isfinite(h0.grad).all()
    for n, p in m.named_parameters():
        assert torch.isfinite(p.grad).all(), n
    capi.device_status()



@pytest.mark.parametrize("shape", [(32, 4, 128, 128), (5, 3, 40, 100), (4, 3, 200, 100)],
                         ids=lambda s: "B%dT%dD%dH%d" % s)
def test_recurrent_gradient_companions_give_up_sets_every_gradient_to_nan(capi_row, shape):
    capi = capi_row
    """At Hp = 128 the module backward forms the recurrent parameter-gradient
    sums in companion workgroups that wait for the chain's alpha/beta words:
    with a budget of 0 they leave at once, and the finalize writes NaN into
    every gradient, dL/dx and dL/dh0; with the default budget again the
    results are finite and the status clean."""
    B1, T1, D1, H1 = shape
    plan = capi.plan(B1, T1, D1, H1, 6)
    assert plan["module_row128_rec_fused"] == 1, plan
    m = _perturbed_module(D1, H1, seed=35).to(DEV)
    x = torch.randn(B1, T1, D1, device=DEV, requires_grad=True)
    h0 = (torch.randn(B1, H1, device=DEV) * 0.2).requires_grad_(True)
    out, (h, _) = m(x, (h0, h0))
    assert torch.isfinite(out).all()
    with _NoWait(capi):
        (out.sum() + h.sum()).backward()
    assert torch.isnan(x.grad).all() and torch.isnan(h0.grad).all()
    for n, p in m.named_parameters():
        assert torch.isnan(p.grad).all(), n
    _expect_fault(capi)
    m.zero_grad(set_to_none=True)
    x.grad = h0.grad = None
    out, (h, _) = m(x, (h0, h0))
    (out.sum() + h.sum()).backward()
    assert torch.isfinite(x.grad).all() and torch.isfinite(h0.grad).all()
    for n, p in m.named_parameters():
        assert torch.isfinite(p.grad).all(), n
    capi.device_status()


# (B, H) whose plan has no clusters of its own: one-row forward clusters, several
# rows per cluster, several launches; chains of 12, 16 and 20 register slots.
AFTER = [(3, 192), (130, 180), (700, 192), (520, 256), (410, 320), (340, 400), (260, 512)]


def _own_kernels(capi, B, H):
    plan = capi.plan(B, T, D, H, 6)
    assert plan["CP"] == 0 and plan["reg_fwd_members"] > 0 and plan["reg_bwd_members"] > 0, plan


def _close(a, b):
    """Two correct float32 evaluations whose sums run in different order."""
    assert torch.isfinite(b).all()
    assert ((a - b).norm() / (a.norm() + 1e-30)).item() <= 1e-5


@pytest.mark.parametrize("B1,H1", AFTER)
def test_sizes_without_own_clusters_complete_after_a_give_up(capi_row, B1, H1):
    """Where the plan has no clusters of its own, the register-resident clusters'
    give-up costs time only: the plan's kernels run behind them, and outputs,
    saved states and gradients are those of the clusters, with a clean status."""
    _own_kernels(capi_row, B1, H1)
    args = boundary(B1, T, D, H1, seed=36)
    g_out, g_h = torch.randn(B1, T, H1, device=DEV), torch.randn(B1, H1, device=DEV)
    ref = None
    for fwd_ok, bwd_ok in ((True, True), (False, True), (True, False), (False, False)):
        with contextlib.nullcontext() if fwd_ok else _NoWait(capi_row):
            dev_args, fwd = gpu_forward(args, save=True)
        with contextlib.nullcontext() if bwd_ok else _NoWait(capi_row):
            grads = gpu_backward(dev_args, fwd[2], g_out, g_h)
        capi_row.device_status()
        res = [*fwd, *grads]
        for a, b in zip(ref or res, res):
            _close(a, b)
        ref = ref or res


@pytest.mark.parametrize("B1,H1", [(3, 192), (130, 180), (520, 256), (410, 320)])
def test_module_path_completes_after_a_give_up(capi_row, B1, H1):
    _own_kernels(capi_row, B1, H1)
    m = _perturbed_module(D, H1, seed=38).to(DEV)
    g = torch.Generator().manual_seed(39)
    x, G = torch.randn(B1, T, D, generator=g), torch.randn(B1, T, H1, generator=g)
    h0 = torch.randn(B1, H1, generator=g) * 0.2
    res = []
    for wait in (True, False):
        m.zero_grad(set_to_none=True)
        xg, hg = x.to(DEV).requires_grad_(True), h0.to(DEV).requires_grad_(True)
        with contextlib.nullcontext() if wait else _NoWait(capi_row):
            out, (h, _) = m(xg, (hg, hg))
            (out * G.to(DEV)).sum().backward()
        res.append([out.detach(), h.detach(), xg.grad, hg.grad, *[q.grad for q in m.parameters()]])
        capi_row.device_status()
    for a, b in zip(*res):
        _close(a, b)


def test_unfold_entry_points_complete_after_a_give_up(capi_row):
    B1, H1 = 5, 192
    _own_kernels(capi_row, B1, H1)
    args = [a.to(DEV) for a in boundary(B1, 1, D, H1, seed=40)]
    M = ltc_cuda._cuda_module
    sens = [torch.randn(B1, H1, device=DEV), torch.rand(B1, H1, device=DEV) * 5]
    ode = [args[1], *args[2:6], *sens, *args[10:13]]
    g_out = torch.randn(B1, H1, device=DEV)
    res = []
    for wait in (True, False):
        with contextlib.nullcontext() if wait else _NoWait(capi_row):
            v, buf = M.ltc_ode_unfold_fwd(*ode, 6, 1e-8, True)
            grads = M.ltc_ode_unfold_bwd(buf, *ode[1:], g_out, 6, 1e-8)
        res.append([v, buf, *grads])
        capi_row.device_status()
    for a, b in zip(*res):
        _close(a, b)


# (B, H, dense): sizes whose plan has clusters, so that a give-up ends in NaN:
# the one-row forward, the two-group forward, the register chain at 16 and 20
# slots and the streaming chain behind it.
OWN = [(3, 320, False), (60, 320, False), (300, 256, False), (2, 512, False), (20, 384, True), (64, 512, True)]


@pytest.mark.parametrize("B1,H1,dense", OWN)
def test_register_clusters_give_up_sets_every_output_to_nan(capi_row, B1, H1, dense):
    plan = capi_row.plan(B1, T, D, H1, 6)
    assert plan["CP"] > 0 and plan["reg_fwd_members"] > 0 and plan["reg_bwd_members"] > 0, plan
    m = _perturbed_module(D, H1, seed=41, sparsity=1.0 if dense else 0.5).to(DEV)
    x = torch.randn(B1, T, D, device=DEV)

    def step(fwd_ok, bwd_ok):
        m.zero_grad(set_to_none=True)
        with contextlib.nullcontext() if fwd_ok else _NoWait(capi_row):
            out, (h, _) = m(x)
        with contextlib.nullcontext() if bwd_ok else _NoWait(capi_row):
            out.sum().backward()
        return [out, h], [q.grad for q in m.parameters()]

    outs, grads = step(False, True)
    assert all(torch.isnan(t).all() for t in outs)
    _expect_fault(capi_row)
    outs, grads = step(True, False)
    assert all(torch.isfinite(t).all() for t in outs)
    assert all(torch.isnan(t).all() for t in grads)
    _expect_fault(capi_row)
    outs, grads = step(True, True)
    assert all(torch.isfinite(t).all() for t in outs + grads)
    capi_row.device_status()


def test_two_streams_at_once(capi_row):
    """Two layers whose plans have no clusters of their own, stepped on two streams
    at the same time: neither can lose its results to the other's workgroups."""
    cases = []
    for i, (B1, H1) in enumerate([(64, 192), (96, 180)]):
        _own_kernels(capi_row, B1, H1)
        m = _perturbed_module(D, H1, seed=42 + i).to(DEV)
        x = torch.randn(B1, 6, D, device=DEV)
        out, _ = m(x)
        out.sum().backward()
        cases.append((m, x, out.detach(), [q.grad.clone() for q in m.parameters()]))
        m.zero_grad(set_to_none=True)
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in cases]
    got = [[], []]
    for _ in range(4):
        for k, (m, x, _, _) in enumerate(cases):
            with torch.cuda.stream(streams[k]):
                out, _ = m(x)
                grads = torch.autograd.grad(out.sum(), list(m.parameters()))
                got[k].append((out.detach(), grads))
    torch.cuda.synchronize()
    for k, (m, x, r_out, r_grads) in enumerate(cases):
        for out, grads in got[k]:
            for a, b in zip([r_out, *r_grads], [out, *grads]):
                _close(a, b)
    capi_row.device_status()
