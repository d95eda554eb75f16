"""The fused z -> (q, k) kernel where several rows share a wavefront (widths 64, 128, 256) and on last
wavefronts that are not full, against float64 with autograd; rel err <= 2e-2."""
import math

import pytest
import torch

from conftest import rel_err
from megalodon_amd import extension as ops
from megalodon_amd.fused_ops import qk_norm_rotary
from megalodon_amd.modules import RotaryEmbedding

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,L,S,Dh,P", [(1, 1, 64, 64, 1), (3, 67, 64, 64, 16), (1, 9, 128, 64, 0), (1, 3, 128, 128, 3),
                                        (2, 1021, 256, 256, 512), (1, 4097, 256, 128, 0), (1, 2, 256, 64, 2)])
def test_narrow_rows_match_float64(B, L, S, Dh, P, dtype):
    g = torch.Generator().manual_seed(S + Dh + L)
    z, dq, dk = ((torch.randn(B, L, S, generator=g) * m).to(dtype) for m in (2, 1, 1))
    gamma, beta = ((torch.randn(2, S, generator=g) * 0.3).to(dtype) for _ in range(2))
    freqs = RotaryEmbedding(Dh, P).get_freqs_cis(0, P) if P else None
    zg, gg, bg = (t.cuda().requires_grad_(True) for t in (z, gamma, beta))
    assert ops.qk_norm_rotary_supported(zg, gg, Dh)
    q, k = qk_norm_rotary(zg, gg, bg, None if freqs is None else freqs.cuda(), Dh, 1e-5)
    torch.autograd.backward((q, k), (dq.cuda(), dk.cuda()))
    z64, g64, b64 = (t.double().requires_grad_(True) for t in (z, gamma, beta))
    zz = z64.view(B, L, S // Dh, Dh)
    zn = (zz * torch.rsqrt(zz.pow(2).mean(-1, keepdim=True) + 1e-5)).view(B, L, S)
    want = list(torch.unbind(zn.unsqueeze(2) * ((g64 + 1.0) / math.sqrt(Dh)) + b64, dim=2))
    if P:
        f = freqs.to(torch.complex128)[torch.arange(L) % P][None, :, None, :]
        want = [torch.view_as_real(torch.view_as_complex(t.reshape(B, L, S // Dh, Dh // 2, 2)) * f).reshape(B, L, S) for t in want]
    torch.autograd.backward(want, (dq.double(), dk.double()))
    for got, ref in ((q, want[0]), (k, want[1]), (zg.grad, z64.grad), (gg.grad, g64.grad), (bg.grad, b64.grad)):
        assert got.dtype == dtype and rel_err(got, ref.detach()) <= 2e-2
