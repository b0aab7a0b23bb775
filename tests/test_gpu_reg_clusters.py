"""The register-resident clusters (128 < H <= 512) against the float64 oracle.

Every rows-per-cluster form at the edges of its range: one row per cluster up
to the last batch that leaves every row a cluster, the two-group form from the
next row on, and the batches that take a second launch; padded and full
columns; recurrent masks with a column that has no synapse, one that has every
synapse and one whose only synapse sits in the last row. The kernels skip
zero-weight synapses but treat a NaN state as the dense kernels they replaced:
it makes every neuron of its row NaN from the next unfold on.
"""

from __future__ import annotations

import pytest
import torch

import ltc_cuda
from _gpu_common import (DEV, _native, _oracle_module_grads, _perturbed_module,  # noqa: F401
                         assert_grads_close, boundary, gpu_backward, gpu_forward,
                         oracle_forward, oracle_grads)

pytestmark = pytest.mark.gpu

# (B, T, D, H, rows per cluster, launches)
FWD = [
    (1, 3, 8, 129, 1, 1),     # Hp = 192: 64-column members, padded columns
    (85, 2, 5, 192, 1, 1),    # 85 clusters of 3 members: the last batch of one row each
    (86, 2, 5, 192, 2, 1),
    (683, 1, 5, 192, 8, 2),   # 680 rows per launch: three rows in the second
    (260, 1, 4, 256, 8, 1),   # Hp = 256 beyond four rows per cluster
    (515, 1, 4, 250, 8, 2),
    (3, 2, 70, 257, 1, 1),    # Hp = 320: 20 synapses per lane at full density
    (52, 2, 5, 320, 4, 1),    # 10 members of 32 columns, 13 clusters
    (21, 2, 5, 380, 1, 1),
    (22, 2, 5, 384, 2, 1),
    (5, 2, 5, 448, 1, 1),
    (16, 1, 5, 512, 1, 1),
    (17, 1, 5, 500, 2, 1),
    (129, 1, 5, 512, 8, 2),
]


def _edge_masks(args):
    """Recurrent columns with no synapse, every synapse, and one in the last row."""
    w_pos, w_erev = args[2], args[3]
    H = w_pos.shape[0]
    w_pos[:, 0] = 0.0
    w_erev[:, 0] = 0.0
    g = torch.Generator().manual_seed(H)
    w_pos[:, H // 2] = torch.rand(H, generator=g) + 0.1
    w_erev[:, H // 2] = w_pos[:, H // 2]
    w_pos[:, H - 1] = 0.0
    w_erev[:, H - 1] = 0.0
    w_pos[H - 1, H - 1] = 0.7
    w_erev[H - 1, H - 1] = -0.7
    return args


@pytest.mark.parametrize("shape", FWD, ids=lambda s: "B%dT%dD%dH%d" % s[:4])
def test_forward_matches_oracle(shape):
    B, T, D, H, rows, launches = shape
    p = ltc_cuda._cuda_module.capi.plan(B, T, D, H, 6)
    assert p["reg_fwd_members"] * p["reg_fwd_cols"] == p["Hp"], p
    assert (p["reg_fwd_rows"], p["reg_fwd_launches"]) == (rows, launches), p
    args = _edge_masks(boundary(B, T, D, H, seed=B + H))
    _, (out, h) = gpu_forward(args)
    ref_out, ref_h = oracle_forward(args)
    err = (out.cpu().double() - ref_out).abs().max().item()
    print(f"{shape}: max|out err| = {err:.2e}", flush=True)
    # float32 sums of up to H terms over T*U unfolds of a contraction: errors of
    # single roundings (6e-8 of values below 1), not the 1e-3 bar
    assert err <= 5e-6
    assert (h.cpu().double() - ref_h).abs().max().item() <= 5e-6


@pytest.mark.parametrize("shape", [(1, 1, 8, 129), (90, 1, 4, 192), (2, 1, 4, 300),
                                   (60, 1, 4, 320), (300, 1, 4, 256)],
                         ids=lambda s: "B%dT%dD%dH%d" % s)
@pytest.mark.parametrize("U", [1, 2, 3])
def test_nan_state_reaches_its_whole_row(shape, U):
    """After one unfold every neuron of the row is NaN, and no other row is."""
    B, T, D, H = shape
    assert ltc_cuda._cuda_module.capi.plan(B, T, D, H, U)["reg_fwd_members"] > 0
    args = boundary(B, T, D, H, seed=13)
    h0 = args[1].clone()
    h0[B - 1, 7] = float("nan")
    _, res = gpu_forward([args[0], h0] + args[2:], U=U)
    out = res[0].cpu()
    assert torch.isnan(out[B - 1]).all()
    assert torch.isfinite(out[:B - 1]).all()


# (B, T, D, H, whether the forward reads the dense image)
@pytest.mark.parametrize("shape", [(1, 5, 8, 192, 0), (1, 1, 8, 192, 1), (90, 1, 4, 192, 0),
                                   (1, 5, 4, 300, 0), (60, 2, 4, 320, 0), (60, 1, 4, 320, 1),
                                   (5, 11, 4, 448, 0), (5, 1, 4, 448, 1), (300, 1, 4, 256, 0)],
                         ids=lambda s: "B%dT%dD%dH%ddense%d" % s)
@pytest.mark.parametrize("i", [0, 7])
def test_infinite_state_saturates_its_gates(shape, i):
    """An infinite v_i makes the gates of its synapses 0 or 1, whatever slot holds
    them or pads a column: every other neuron stays finite and equals the oracle."""
    B, T, D, H, dense = shape
    p = ltc_cuda._cuda_module.capi.plan(B, T, D, H, 6)
    assert p["reg_fwd_members"] > 0 and p["reg_fwd_dense"] == dense
    args = _edge_masks(boundary(B, T, D, H, seed=14))
    h0 = args[1].clone()
    h0[0, i] = float("inf")
    h0[B - 1, i] = -float("inf")
    _, (out, h) = gpu_forward([args[0], h0] + args[2:])
    ref_out, ref_h = oracle_forward([args[0], h0] + args[2:])
    keep = [j for j in range(H) if j != i]
    for got, ref in ((out, ref_out), (h, ref_h)):
        got = got.cpu().double()[..., keep]
        assert torch.isfinite(ref[..., keep]).all()
        # the bound of test_forward_matches_oracle
        assert (got - ref[..., keep]).abs().max().item() <= 5e-6


@pytest.mark.parametrize("shape", [(2, 1, 4, 192), (2, 30, 4, 192), (90, 1, 4, 192), (2, 1, 4, 320),
                                   (2, 30, 4, 320), (60, 1, 4, 320), (60, 10, 4, 320),
                                   (300, 1, 4, 256)],
                         ids=lambda s: "B%dT%dD%dH%d" % s)
@pytest.mark.parametrize("leaf,value", [("mu", float("nan")), ("sigma", float("nan")),
                                        ("mu", float("inf"))])
def test_non_finite_operand_at_a_masked_synapse(shape, leaf, value):
    """Masked or not, a synapse with a NaN gate makes its neuron NaN (0 * NaN), and
    one with an infinite argument does not (0 * 0 or 0 * 1): the output and
    dL/dh0 are finite exactly where the oracle has them so."""
    B, T, D, H = shape
    m = _perturbed_module(D, H, seed=6).to(DEV)
    m.ode_unfolds = 1
    p = ltc_cuda._cuda_module.capi.plan(B, T, D, H, 1)
    assert p["reg_fwd_members"] > 0 and p["reg_fwd_dense"] == (T == 1 and B < 90)
    with torch.no_grad():
        m.sparsity_mask[5, 9] = m.sparsity_mask[H - 1, H - 1] = 0.0
        getattr(m, leaf)[5, 9] = value
        getattr(m, leaf)[H - 1, H - 1] = -value
    g = torch.Generator().manual_seed(2)
    x = torch.randn(B, T, D, generator=g)
    h0 = torch.randn(B, H, generator=g) * 0.2
    hg = h0.to(DEV).requires_grad_(True)
    out, (h, _) = m(x.to(DEV), (hg, hg))
    out.sum().backward()
    r_out, _, _, _, r_gh = _oracle_module_grads(m, x, h0, torch.ones(B, T, H), torch.zeros(B, H))
    assert torch.equal(torch.isfinite(out.cpu()), torch.isfinite(r_out))
    assert torch.equal(torch.isfinite(hg.grad.cpu()), torch.isfinite(r_gh))


def test_nan_sum_spreads_one_unfold_later():
    """A NaN input at a neuron's sensory synapse makes that neuron NaN in the
    first unfold and its whole row NaN in the second, as a dense kernel does."""
    B, T, D, H = 60, 1, 6, 320
    args = boundary(B, T, D, H, seed=3)
    x = args[0].clone()
    x[2, 0, 1] = float("nan")
    connected = args[9][1] != 0  # sensory_w_pos[d = 1]
    _, res = gpu_forward([x] + args[1:], U=1)
    assert torch.equal(torch.isnan(res[0].cpu()[2, 0]), connected)
    _, res = gpu_forward([x] + args[1:], U=2)
    assert torch.isnan(res[0].cpu()[2, 0]).all()
    assert torch.isfinite(res[0].cpu()[3]).all()


# (B, T, D, H, density, rows per cluster, launches): the chain, which needs
# 16 (H <= 448) or 20 synapses per thread and past that runs the kernel that
# streams dense operands
BWD = [
    (1, 3, 8, 129, 0.5, 2, 1),
    (85, 2, 5, 192, 0.5, 4, 1),
    (337, 1, 5, 192, 1.0, 8, 2),   # 336 rows per launch; 12 synapses each when dense
    (257, 1, 4, 256, 0.5, 8, 2),   # one row in the second launch
    (3, 2, 70, 257, 0.5, 2, 1),
    (101, 1, 5, 320, 0.5, 8, 1),   # 4 gather words per thread
    (30, 2, 5, 320, 1.0, 2, 1),    # streamed
    (43, 2, 5, 384, 0.5, 4, 1),    # 21 clusters of 12 members hold 42 rows at two each
    (22, 1, 5, 384, 1.0, 2, 1),
    (150, 1, 5, 448, 1.0, 8, 2),
    (37, 1, 5, 448, 0.5, 4, 1),
    (129, 1, 5, 512, 0.5, 8, 2),
    (40, 1, 5, 500, 1.0, 4, 1),
]


@pytest.mark.parametrize("shape", BWD, ids=lambda s: "B%dT%dD%dH%dp%g" % s[:5])
def test_module_backward_matches_oracle(shape):
    B, T, D, H, density, rows, launches = shape
    p = ltc_cuda._cuda_module.capi.plan(B, T, D, H, 6)
    assert p["reg_bwd_members"] * 32 == p["Hp"], p
    assert (p["reg_bwd_rows"], p["reg_bwd_launches"]) == (rows, launches), p
    m = _perturbed_module(D, H, seed=B + H, sparsity=density).to(DEV)
    with torch.no_grad():  # a neuron whose only outgoing synapse ends at the last one
        m.sparsity_mask[2] = 0.0
        m.sparsity_mask[2, H - 1] = 1.0
    g = torch.Generator().manual_seed(17)
    x = torch.randn(B, T, D, generator=g)
    h0 = torch.randn(B, H, generator=g) * 0.2
    G = torch.randn(B, T, H, generator=g)
    Gh = torch.randn(B, H, generator=g)
    xg = x.to(DEV).requires_grad_(True)
    hg = h0.to(DEV).requires_grad_(True)
    out, (h, _) = m(xg, (hg, hg))
    ((out * G.to(DEV)).sum() + (h * Gh.to(DEV)).sum()).backward()
    r_out, r_h, r_g, r_gx, r_gh = _oracle_module_grads(m, x, h0, G, Gh)
    # float32 sums over U*T*B instances in fixed order: relative 2-norm errors
    # of a few 1e-6; 2e-5 leaves the room the weight gradients' cancelling
    # terms need
    for name, a, b in ([("x", xg.grad, r_gx), ("h0", hg.grad, r_gh)]
                       + [(n, q.grad, r_g[n]) for n, q in m.named_parameters()]):
        err = ((a.cpu().double() - b).norm() / b.norm()).item()
        assert err <= 2e-5, f"{name}: {err:.1e}"


@pytest.mark.parametrize("shape", [(5, 2, 6, 192), (300, 1, 4, 256), (40, 1, 4, 320),
                                   (20, 2, 4, 500)], ids=lambda s: "B%dT%dD%dH%d" % s)
def test_boundary_backward_with_unequal_zero_weights(shape):
    """w_pos = 0 where w_erev is not (and the other way round): the factor the
    register form takes out of them does not exist there."""
    B, T, D, H = shape
    assert ltc_cuda._cuda_module.capi.plan(B, T, D, H, 6)["reg_bwd_members"] > 0
    args = boundary(B, T, D, H, seed=5)
    g = torch.Generator().manual_seed(6)
    pick = torch.rand(H, H, generator=g)
    args[2] = torch.where(pick < 0.1, torch.zeros(()), args[2])
    args[3] = torch.where(pick > 0.9, torch.zeros(()), args[3])
    dev_args, (out, h, saved) = gpu_forward(args, save=True)
    g_out = torch.randn(B, T, H, generator=g)
    g_h = torch.randn(B, H, generator=g)
    got = gpu_backward(dev_args, saved, g_out.to(DEV), g_h.to(DEV))
    ref = oracle_grads(args, g_out, g_h)
    assert_grads_close(got, ref, f"{shape}")


@pytest.mark.parametrize("shape", [(6, 1, 4, 192), (60, 1, 4, 384)],
                         ids=lambda s: "B%dT%dD%dH%d" % s)
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_non_finite_gradient_reaches_its_whole_row(shape, value):
    """Zero weight times a non-finite dL/dout is NaN: dL/dh0 of that row has no
    finite entry, and every other row is untouched."""
    B, T, D, H = shape
    m = _perturbed_module(D, H, seed=4).to(DEV)
    x = torch.randn(B, T, D, generator=torch.Generator().manual_seed(1)).to(DEV)
    h0 = torch.zeros(B, H, device=DEV, requires_grad=True)
    out, _ = m(x, (h0, h0))
    G = torch.ones(B, T, H, device=DEV)
    clean, = torch.autograd.grad(out, h0, G, retain_graph=True)
    G[3, 0, 11] = value
    dirty, = torch.autograd.grad(out, h0, G)
    assert not torch.isfinite(dirty[3]).any()
    keep = [b for b in range(B) if b != 3]
    assert torch.equal(dirty[keep], clean[keep])


@pytest.mark.parametrize("shape", [(5, 2, 6, 192), (40, 3, 4, 320)], ids=lambda s: "B%dT%dD%dH%d" % s)
@pytest.mark.parametrize("sigma,mu", [(0.0, 0.5), (1e-22, 0.5), (1e-22, 1e22), (-1e-21, 2e21),
                                      (1e-15, 1e15)])
def test_gradients_at_a_vanishing_slope(shape, sigma, mu):
    """A slope too small to tell the states apart: the gate is 1/2, or that of the
    offset alone when |mu| is as large as the slope is small."""
    B, T, D, H = shape
    m = _perturbed_module(D, H, seed=8).to(DEV)
    with torch.no_grad():
        m.sparsity_mask[3, 4] = 1.0
        m.sigma[3, 4], m.mu[3, 4] = sigma, mu
    g = torch.Generator().manual_seed(9)
    x = torch.randn(B, T, D, generator=g)
    h0 = torch.randn(B, H, generator=g) * 0.2
    G = torch.randn(B, T, H, generator=g)
    hg = h0.to(DEV)
    out, _ = m(x.to(DEV), (hg, hg))
    (out * G.to(DEV)).sum().backward()
    _, _, r_g, _, _ = _oracle_module_grads(m, x, h0, G, torch.zeros(B, H))
    for n in ("w", "erev", "mu", "sigma"):
        got = dict(m.named_parameters())[n].grad[3, 4].item()
        ref = r_g[n][3, 4].item()
        # a float32 sum of a few hundred terms whose signs differ
        assert abs(got - ref) <= 1e-4 * abs(ref) + 1e-30, (n, got, ref)


@pytest.mark.parametrize("shape", [(2, 100, 8, 192, 0.5), (2, 100, 8, 192, 1.0), (2, 100, 8, 320, 0.5),
                                   (3, 60, 8, 320, 1.0), (1, 100, 8, 448, 0.5), (2, 60, 8, 512, 1.0)],
                         ids=lambda s: "B%dT%dD%dH%dp%g" % s)
def test_gradient_sums_of_long_sequences(shape):
    """Hundreds of unfolds of a few rows: the recurrent sums move out of the
    registers on the way, so their error is that of sums of some 50 terms and of
    as many such sums (2.1 to 3.3e-7; 4.6 to 10e-7 in one sum each)."""
    B, T, D, H, density = shape
    p = ltc_cuda._cuda_module.capi.plan(B, T, D, H, 6)
    assert 0 < p["reg_bwd_move"] < T * 6
    m = _perturbed_module(D, H, seed=B + H, sparsity=density).to(DEV)
    g = torch.Generator().manual_seed(21)
    x = torch.randn(B, T, D, generator=g)
    h0 = torch.randn(B, H, generator=g) * 0.2
    G = torch.randn(B, T, H, generator=g)
    hg = h0.to(DEV)
    out, _ = m(x.to(DEV), (hg, hg))
    (out * G.to(DEV)).sum().backward()
    _, _, r_g, _, _ = _oracle_module_grads(m, x, h0, G, torch.zeros(B, H))
    for n in ("w", "erev", "mu"):
        q = dict(m.named_parameters())[n].grad.cpu().double()
        err = ((q - r_g[n]).norm() / r_g[n].norm()).item()
        print(f"{shape} {n}: {err:.2e}", flush=True)
        assert err <= 4.3e-7, f"{n}: {err:.1e}"


# (B, T, D, H, density, dense forward, dense chain, register chain): both sides of
# the rules for the image that forward and chain read, and of the slot limit
IMAGES = [(1, 4, 8, 192, 0.5, 1, 0, 1), (1, 5, 8, 192, 0.5, 0, 0, 1), (86, 1, 5, 130, 0.5, 0, 0, 1),
          (3, 2, 70, 257, 0.5, 1, 1, 0), (3, 3, 70, 257, 0.5, 1, 0, 1), (3, 5, 70, 257, 0.5, 0, 0, 1),
          (52, 1, 5, 320, 0.5, 1, 1, 0), (52, 2, 5, 320, 0.5, 0, 0, 1), (52, 2, 5, 320, 1.0, 0, 0, 0),
          (5, 10, 5, 400, 0.5, 1, 0, 1), (5, 11, 5, 400, 0.5, 0, 0, 1), (9, 3, 5, 500, 0.5, 1, 0, 1),
          (33, 1, 5, 512, 0.5, 1, 1, 0), (33, 2, 5, 512, 0.5, 0, 0, 1)]


@pytest.mark.parametrize("shape", IMAGES, ids=lambda s: "B%dT%dD%dH%dp%g" % s[:5])
def test_dense_and_compacted_images(shape):
    B, T, D, H, density, df, db, reg = shape
    p = ltc_cuda._cuda_module.capi.plan(B, T, D, H, 6)
    assert (p["reg_fwd_dense"], p["reg_bwd_dense"]) == (df, db), p
    m = _perturbed_module(D, H, seed=B + T, sparsity=density).to(DEV)
    # the register chain takes columns (rows of the mask) of at most 16 slots a
    # thread in 16 chunks, 20 above Hp = 448
    limit = p["Hp"] if p["Hp"] <= 256 else (256 if p["Hp"] <= 448 else 320)
    fits = int((m.sparsity_mask != 0).sum(1).max()) <= limit
    assert reg == (fits and not db)
    g = torch.Generator().manual_seed(23)
    x = torch.randn(B, T, D, generator=g)
    h0 = torch.randn(B, H, generator=g) * 0.2
    G = torch.randn(B, T, H, generator=g)
    xg, hg = x.to(DEV).requires_grad_(True), h0.to(DEV).requires_grad_(True)
    out, _ = m(xg, (hg, hg))
    (out * G.to(DEV)).sum().backward()
    r_out, _, r_g, r_gx, r_gh = _oracle_module_grads(m, x, h0, G, torch.zeros(B, H))
    assert (out.detach().cpu().double() - r_out).abs().max().item() <= 5e-6
    for name, a, b in ([("x", xg.grad, r_gx), ("h0", hg.grad, r_gh)]
                       + [(n, q.grad, r_g[n]) for n, q in m.named_parameters()]):
        err = ((a.cpu().double() - b).norm() / b.norm()).item()
        assert err <= 2e-5, f"{name}: {err:.1e}"


@pytest.mark.parametrize("shape", [(2, 3, 8, 192), (64, 2, 8, 320), (40, 1, 8, 500), (3, 10, 4, 512)],
                         ids=lambda s: "B%dT%dD%dH%d" % s)
def test_boundary_gradients(shape):
    """A backward over the boundary tensors wants every synapse's gradients: dense
    columns, whatever the image rule says."""
    B, T, D, H = shape
    args = _edge_masks(boundary(B, T, D, H, seed=7))
    dev_args, (out, h, saved) = gpu_forward(args, save=True)
    g = torch.Generator().manual_seed(8)
    g_out, g_h = torch.randn(B, T, H, generator=g), torch.randn(B, H, generator=g)
    got = gpu_backward(dev_args, saved, g_out.to(DEV), g_h.to(DEV))
    assert_grads_close(got, oracle_grads(args, g_out, g_h), f"{shape}")


@pytest.mark.parametrize("shape", [(60, 2, 4, 384), (6, 3, 4, 320)], ids=lambda s: "B%dT%dD%dH%d" % s)
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_non_finite_gradient_in_the_compacted_chain(shape, value):
    """As test_non_finite_gradient_reaches_its_whole_row, at the last of several
    steps."""
    B, T, D, H = shape
    assert ltc_cuda._cuda_module.capi.plan(B, T, D, H, 6)["reg_bwd_dense"] == 0
    m = _perturbed_module(D, H, seed=4).to(DEV)
    x = torch.randn(B, T, D, generator=torch.Generator().manual_seed(1)).to(DEV)
    h0 = torch.zeros(B, H, device=DEV, requires_grad=True)
    out, _ = m(x, (h0, h0))
    G = torch.ones(B, T, H, device=DEV)
    clean, = torch.autograd.grad(out, h0, G, retain_graph=True)
    G[3, T - 1, 0] = value
    dirty, = torch.autograd.grad(out, h0, G)
    assert not torch.isfinite(dirty[3]).any()
    keep = [b for b in range(B) if b != 3]
    assert torch.equal(dirty[keep], clean[keep])


@pytest.mark.parametrize("shape", [(6, 4, 5, 320), (6, 4, 5, 512)], ids=lambda s: "B%dT%dD%dH%d" % s)
def test_a_weight_that_cannot_be_factored_out_takes_the_streaming_chain(shape):
    """|erev| above 1e18 at a weight of e^-80: a synapse worth 1e-17, so every other
    gradient is the same to a rounding, but the register chain, which divides by
    the weight, may not run. Which one ran shows in the last bits."""
    B, T, D, H = shape
    assert ltc_cuda._cuda_module.capi.plan(B, T, D, H, 6)["reg_bwd_dense"] == 0
    m = _perturbed_module(D, H, seed=12).to(DEV)
    with torch.no_grad():
        m.sparsity_mask[6, 5] = 1.0
        m.w[6, 5] = -80.0
    x = torch.randn(B, T, D, generator=torch.Generator().manual_seed(2)).to(DEV)
    h0 = torch.zeros(B, H, device=DEV)
    res = []
    for erev in (1.0, 5e17, 2e18):
        with torch.no_grad():
            m.erev[6, 5] = erev
        m.zero_grad(set_to_none=True)
        out, _ = m(x, (h0, h0))
        out.sum().backward()
        gs = [m.mu.grad.clone(), m.sigma.grad.clone(), m.erev.grad.clone()]
        for t in gs:
            t[6, 5] = 0.0
        res.append(gs)
    one, below, above = res
    for a, b, c in zip(one, below, above):
        assert torch.equal(a, b)
        assert not torch.equal(a, c)
        assert ((a - c).norm() / a.norm()).item() <= 1e-5
