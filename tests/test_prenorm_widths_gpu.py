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


@pytest.mark.parametrize("k,f32", [(5376, False), (5376, True), (1536, False), (1536, True)])
def test_prenorm_straight_rows_match_general_path(device, k, f32):
    """The straight-line rows against the general kernel, which the same values take where the table
    rows are not 16-byte aligned: the same bytes, flags among them, for strided rows, a table row per
    row and rows of zeros, subnormals, the largest bf16 (their sum of squares overflows), inf and NaN.
    At 5376 columns both order the sum of squares alike. At 1536 the general kernel's order is
    another: there the values are small integers, whose squares sum exactly in any order."""
    rows = 203
    g = torch.Generator().manual_seed(k + f32)
    dt = torch.float32 if f32 else torch.bfloat16
    if k == 5376:
        x = torch.randn(rows, k, generator=g) * 2.0 ** torch.randint(-8, 9, (1, k), generator=g)
    else:
        x = torch.randint(-8, 9, (rows, k), generator=g).float()
    x[3], x[4], x[5] = 0.0, 2.0 ** -130, 3.3e38
    x[6, k - 1], x[7, 0], x[8, k // 2] = float("inf"), -float("inf"), float("nan")
    store = torch.zeros(rows, k + 64, dtype=torch.bfloat16, device=device)
    store[:, :k] = x.to(torch.bfloat16).to(device)
    x = store[:, :k]
    w = (1 + 0.1 * torch.randn(k, generator=g)).to(dt).to(device)
    tables = (torch.randn(2, 5, k, generator=g) * 0.3).to(dt).to(device)
    loose = torch.zeros(2, 5, k + 1, dtype=dt, device=device)
    loose[:, :, :k] = tables
    idx = (torch.arange(rows) % 5).to(device)
    a = vm.launch_prenorm_quantize(x, w, 1e-6, tables[0], tables[1], idx, write_bf16=True)
    b = vm.launch_prenorm_quantize(x, w, 1e-6, loose[0, :, :k], loose[1, :, :k], idx, write_bf16=True)
    assert a[3].cpu().tolist() == [r not in (6, 7, 8) for r in range(a[3].shape[0])]
    bits = lambda t: t.view(torch.int16) if t.dtype == torch.bfloat16 else t
    for name, p, q in zip(("bf16", "codes", "scales", "finite"), a, b):
        assert torch.equal(bits(p), bits(q)), name
