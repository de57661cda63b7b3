"""The prenorm producer's straight-line rows at the widths with a half slice (5376 = 10.5 x 512
columns) and an odd slice count (1536), against the oracle: rows sharing a table row, groups of
them, mixed, and fp32 tables; the padding rows' codes, scales and flags."""
import numpy as np
import pytest
import torch

from oracle import mxfp8 as om
from vdn_amd import mxfp8 as vm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,k,pattern,f32", [(1, 5376, "shared", False), (300, 5376, "groups", False),
                                                 (260, 5376, "mixed", True), (129, 1536, "shared", True),
                                                 (77, 1536, "mixed", False)])
def test_prenorm_half_slice_widths(device, rows, k, pattern, f32):
    g = torch.Generator().manual_seed(rows + k)
    dt = torch.float32 if f32 else torch.bfloat16
    x = (torch.randn(rows, k, generator=g) * 2).to(torch.bfloat16)
    w = (1 + 0.1 * torch.randn(k, generator=g)).to(dt)
    scale, shift = ((torch.randn(5, k, generator=g) * 0.3).to(dt) for _ in range(2))
    idx = {"shared": torch.full((rows,), 2), "groups": torch.arange(rows) // 64 % 5,
           "mixed": torch.arange(rows) % 5}[pattern].long()
    y, q, s, finite = vm.launch_prenorm_quantize(x.to(device), w.to(device), 1e-6, scale.to(device),
                                                 shift.to(device), idx.to(device), write_bf16=True)
    ref, mag = om.prenorm(x.float().numpy(), w.float().numpy(), 1e-6, scale.float().numpy(),
                          shift.float().numpy(), idx.numpy(), return_magnitude=True)
    yc = y.float().cpu().numpy()
    # one bf16 ulp, or a few fp32 ulps of the addends where they cancel
    assert (np.abs(yc - ref) <= om.bf16_ulp(ref) + 2.0 ** -21 * mag).all()
    assert (yc == ref).mean() > 0.999
    codes, _, flat = om.quantize(yc)
    assert np.array_equal(q.cpu().numpy(), codes) and np.array_equal(s.cpu().numpy(), flat)
    assert bool(finite.all()) and finite.shape == (q.shape[0],)
    x[rows - 1, k - 1] = float("inf")
    _, q2, s2, f2 = vm.launch_prenorm_quantize(x.to(device), w.to(device), 1e-6, scale.to(device),
                                               shift.to(device), idx.to(device), write_bf16=False)
    assert torch.equal(q2[:rows - 1], q[:rows - 1])
    assert f2.cpu().tolist() == [r != rows - 1 for r in range(q.shape[0])]
