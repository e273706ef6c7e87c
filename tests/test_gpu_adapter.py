"""GPU parity of the fused residual output adapter (sva_residual_adapter)
against the float64 oracle of experiments/sva_late4_logit_distill.py:47-51:
within 1e-5 of the output's magnitude for fp32 activations, 2e-2 for bf16
(the correction is cast to the attention dtype before the residual add, as
the reference does); token counts that do not fill a workgroup; the module
wrapper end to end; inference only."""

from __future__ import annotations

import numpy as np
import pytest
import torch
from torch import nn

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,H,rank,dtype", [(1, 576, 16, torch.float32), (37, 576, 16, torch.float32),
                                            (8, 576, 16, torch.bfloat16), (1000, 64, 5, torch.bfloat16),
                                            (3, 2048, 64, torch.float32)])
def test_residual_adapter_matches_oracle(device, T, H, rank, dtype):
    from sva_amd import kernels

    rng = np.random.default_rng(T + H + rank)
    hidden = rng.standard_normal((T, H)).astype(np.float32)
    attn = rng.standard_normal((T, H)).astype(np.float32)
    down = (rng.standard_normal((rank, 2 * H)) * 0.02).astype(np.float32)
    up = (rng.standard_normal((H, rank)) * 0.5).astype(np.float32)
    h = torch.from_numpy(hidden).to(device, dtype)
    a = torch.from_numpy(attn).to(device, dtype)
    out = kernels.residual_adapter(h, a, torch.from_numpy(down).to(device), torch.from_numpy(up).to(device), 0.75)
    assert out.dtype == dtype and out.shape == a.shape
    ref = oracle.residual_adapter(h.float().cpu().numpy(), a.float().cpu().numpy(), down, up, 0.75)
    got = out.float().cpu().numpy()
    tol = 1e-5 if dtype == torch.float32 else 2e-2
    err = np.abs(got - ref).max() / np.abs(ref).max()
    assert err <= tol, f"rel err {err}"


@pytest.mark.parametrize("T,H,rank,dtype,odd", [
    (1, 5, 1, torch.float32, False),        # fewer inputs than lanes
    (257, 130, 7, torch.float16, False),    # two tokens a workgroup, the last alone; rows of 260 inputs
    (1025, 576, 20, torch.float32, False),  # four to eight tokens a workgroup, a rank past the prefetched weights
    (2049, 576, 16, torch.bfloat16, True),  # weights at odd addresses
    (2, 1500, 64, torch.float32, False),    # more outputs than threads
    (3, 8192, 3, torch.float32, False),     # the widest model
])
def test_adapter_workgroup_shapes(device, T, H, rank, dtype, odd):
    """Every token count a workgroup takes and both weight layouts, against float64: sums of at most 2 H + rank
    fp32 products in any order are within (2 H + rank) 2^-24 of their absolute sum, far inside 1e-5."""
    from sva_amd import kernels

    g = torch.Generator(device=device).manual_seed(T + H)
    h = torch.randn(T, H, device=device, generator=g).to(dtype)
    a = torch.randn(T, H, device=device, generator=g).to(dtype)

    def weight(rows, cols, std):
        w = torch.randn(rows, cols, device=device, generator=g) * std
        if not odd:
            return w
        buf = torch.empty(rows * cols + 1, device=device)[1:].view(rows, cols)
        return buf.copy_(w)

    down, up = weight(rank, 2 * H, 0.02), weight(H, rank, 0.5)
    out = kernels.residual_adapter(h, a, down, up, 0.75)
    x = torch.cat([h, a], -1).double()
    corr = torch.nn.functional.gelu(x @ down.double().T) @ up.double().T * 0.75
    ref = a.double() + corr.to(dtype).double()
    err = float((out.double() - ref).abs().max() / ref.abs().max())
    assert err <= {torch.float32: 1e-5, torch.float16: 2e-3, torch.bfloat16: 2e-2}[dtype], f"rel err {err}"


@pytest.mark.parametrize("T,H", [(3, 576), (300, 576), (2, 130), (1, 8192)])
def test_adapter_keeps_an_infinity(device, T, H):
    """An infinity among a token's last attention values meets its own weights only: with positive weights for it,
    every output of that token is +infinity (never a NaN) and the other tokens' outputs are what they are without it."""
    from sva_amd import kernels

    g = torch.Generator(device=device).manual_seed(H)
    h, a = (torch.randn(T, H, device=device, generator=g) for _ in range(2))
    down, up = torch.rand(4, 2 * H, device=device, generator=g) + 0.1, torch.rand(H, 4, device=device, generator=g) + 0.1
    plain = kernels.residual_adapter(h, a, down, up, 1.0)
    a[T // 2, H - 2] = float("inf")
    out = kernels.residual_adapter(h, a, down, up, 1.0)
    assert bool((out[T // 2] == float("inf")).all())
    rest = torch.arange(T, device=device) != T // 2
    assert torch.equal(out[rest], plain[rest])


class _Fixed(nn.Module):
    def __init__(self, out):
        super().__init__()
        self.out = out

    def forward(self, hidden_states, *args, **kwargs):
        return self.out, None


def test_adapter_module_wraps_attention(device):
    from sva_amd.adapter import SVAResidualOutputAdapter

    rng = np.random.default_rng(2)
    hidden = torch.from_numpy(rng.standard_normal((1, 5, 576)).astype(np.float32)).to(device, torch.bfloat16)
    attn = torch.from_numpy(rng.standard_normal((1, 5, 576)).astype(np.float32)).to(device, torch.bfloat16)
    mod = SVAResidualOutputAdapter(_Fixed(attn), 576, 16, 1.0).to(device)
    with torch.no_grad():
        out, weights = mod(hidden)
        assert weights is None
        assert torch.equal(out, attn)  # zero-initialised up projection
        mod.up.weight.normal_(std=0.5)
        out, _ = mod(hidden)
    ref = oracle.residual_adapter(hidden[0].float().cpu().numpy(), attn[0].float().cpu().numpy(),
                                  mod.down.weight.detach().cpu().numpy(), mod.up.weight.detach().cpu().numpy(), 1.0)
    err = np.abs(out[0].float().cpu().numpy() - ref).max() / np.abs(ref).max()
    assert err <= 2e-2
    with pytest.raises(RuntimeError, match="inference only"):
        mod(hidden)  # gradients enabled and trainable weights
