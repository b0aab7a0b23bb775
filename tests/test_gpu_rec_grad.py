"""The recurrent parameter-gradient pass of unfused chains over the unmasked
synapses only: tiles of 32 x 64 synapses listed (up to 1536 entries) or, nearly
full, evaluated whole; tiles with no synapse, with one, at the padding of H, and
one to six slots per thread, against the float64 oracle."""

from __future__ import annotations

import pytest
import torch

import ltc_cuda
from _gpu_common import DEV, _native, _oracle_module_grads, _perturbed_module  # noqa: F401

pytestmark = pytest.mark.gpu

# (B, T, D, H, density)
SHAPES = [(65, 1, 5, 65, 0.5), (70, 2, 9, 100, 0.1), (66, 2, 5, 128, 0.3), (66, 2, 5, 128, 0.72),
          (66, 1, 5, 128, 0.9), (65, 1, 5, 128, 1.0), (2, 2, 5, 600, 0.5), (1, 1, 4, 577, 1.0)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "B%dT%dD%dH%dp%g" % s)
def test_gradients_match_oracle(shape):
    B, T, D, H, density = shape
    p = ltc_cuda._cuda_module.capi.plan(B, T, D, H, 6)
    assert p["fuse"] == 0 and p["module_row128_rec_fused"] == 0 and p["reg_bwd_members"] == 0
    m = _perturbed_module(D, H, seed=B + H, sparsity=density).to(DEV)
    with torch.no_grad():
        m.sparsity_mask[:32, :64] = 0.0   # a tile with no synapse but one
        m.sparsity_mask[31, 63] = 1.0
        m.sparsity_mask[32:64, 64:] = 0.0  # (and none at all)
    g = torch.Generator().manual_seed(3)
    x = torch.randn(B, T, D, generator=g)
    h0 = torch.randn(B, H, generator=g) * 0.2
    G = torch.randn(B, T, H, generator=g)
    xg = x.to(DEV).requires_grad_(True)
    hg = h0.to(DEV)
    out, _ = m(xg, (hg, hg))
    (out * G.to(DEV)).sum().backward()
    _, _, r_g, _, _ = _oracle_module_grads(m, x, h0, G, torch.zeros(B, H))
    for n in ("w", "erev", "mu", "sigma"):
        q = dict(m.named_parameters())[n].grad.cpu().double()
        # masked synapses exactly zero; the rest a few float32 roundings of sums
        # whose terms may cancel
        assert (q[m.sparsity_mask.cpu() == 0] == 0).all(), n
        err = ((q - r_g[n]).norm() / r_g[n].norm()).item()
        assert err <= 2e-5, f"{n}: {err:.1e}"
