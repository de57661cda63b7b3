"""The block-scaled GEMM's planned kernels (the stream kernel of the small and middle sizes, the large
kernel, and both in one call) against the oracle.

Each shape names the kernels it is there for, and the test asserts that the plan takes them: the
stream kernel's 128- and 256-column tiles, one and several tiles per workgroup, the rows left below
whole waves of the large kernel, padded columns past the last 256-column tile, single and odd K steps
and the last partial rows. Each is checked on sampled rows against the exactly dequantized float64
GEMM, within the accumulation bound of tests/test_mxfp8_gpu.py::test_gemm_gated_residual_epilogue,
for the bf16, gated-residual and producer epilogues.
"""
import ctypes

import numpy as np
import pytest
import torch

from oracle import mxfp8 as om
from vdn_amd import _lib
from vdn_amd import mxfp8 as vm

pytestmark = pytest.mark.gpu

# (m, n, k, rows of the large kernel, columns of the stream kernel's tiles below them)
SHAPES = [
    (1, 128, 128, 0, 128),         # one tile, one K step
    (77, 5120, 1152, 0, 128),      # few tiles, 9 K steps
    (130, 200, 384, 0, 128),       # an odd number of steps, n below its padding
    (300, 1920, 640, 0, 128),
    (512, 5120, 1024, 0, 128),
    (1560, 5120, 256, 0, 128),     # two whole rounds of the CUs and a third, partial one
    (960, 5120, 768, 0, 256),      # one tile each
    (960, 5200, 768, 0, 256),      # padded N 5248: the last 256-column tile half past it
    (2304, 7168, 384, 0, 256),     # a whole round and a partial one
    (2040, 8192, 1280, 2048, 0),   # the large kernel, the last rows past M
    (2177, 8192, 2304, 2048, 128),  # the large kernel, then the rows below its whole wave
    (4097, 5376, 3712, 3072, 256),
]


def assert_plan(m, n, k, kind, large_rows, tile_cols):
    """The kernels the size takes on this device, so that another choice cannot leave one untested."""
    rows, cols = ctypes.c_int64(-1), ctypes.c_int(-1)
    _lib.call("vdn_mxfp8_gemm_plan", -(-m // 128) * 128, -(-n // 128) * 128, -(-k // 128) * 128, kind,
              ctypes.byref(rows), ctypes.byref(cols))
    assert (rows.value, cols.value) == (large_rows, tile_cols)


def operands(m, n, k):
    g = torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16)
    w = (torch.randn(n, k, generator=g) * 0.05).to(torch.bfloat16)
    bias = (torch.randn(n, generator=g) * 0.5).to(torch.bfloat16)
    gate = torch.randn(n, generator=g).to(torch.bfloat16)
    res = torch.randn(m, n, generator=g).to(torch.bfloat16)
    rows = np.unique(np.concatenate([np.arange(0, m, 128), np.arange(127, m, 128),
                                     np.arange(max(0, m - 3), m)]))
    wc, wn, _ = om.quantize(w.float().numpy())
    ac, an, _ = om.quantize(x[torch.from_numpy(rows)].float().numpy())
    y0 = om.bf16_round(om.gemm(ac, an, wc, wn, len(rows), n))
    mag = om.gemm_magnitude(ac, an, wc, wn, len(rows), n)
    y = om.bf16_round(y0 + bias.float().numpy()[None])
    limit = om.bf16_ulp(y0) + om.bf16_ulp(y) + om.MFMA_ACCUMULATION_BOUND * mag
    return x, w, bias, gate, res, rows, y, limit


def check(got, rows, ref, limit):
    got = got[torch.from_numpy(rows).to(got.device)].float().cpu().numpy().astype(np.float64)
    err = np.abs(got - ref)
    assert (err <= limit).all(), float((err / limit).max())


@pytest.mark.parametrize("m,n,k,large_rows,tile_cols", SHAPES)
def test_stream_gemm_matches_oracle(device, m, n, k, large_rows, tile_cols):
    for kind in range(3):
        assert_plan(m, n, k, kind, large_rows, tile_cols)
    x, w, bias, gate, res, rows, y, limit = operands(m, n, k)
    q, s = vm.quantize_activation(x.to(device))
    wq, ws = vm.quantize_activation(w.to(device))
    b, g = bias.to(device), gate.to(device)
    flag = torch.zeros(1, dtype=torch.int32, device=device)
    store = torch.full((m + 5, n), 7.0, dtype=torch.bfloat16, device=device)
    plain = vm.mxfp8_gemm(q, s, wq, ws, n, rows=m, bias=b, out=store[:m], nonfinite=flag)
    assert bool((store[m:] == 7.0).all()), "rows past M are not written"
    check(plain, rows, y, limit)
    # gated residual, over the residual itself
    out = res.to(device)
    vm.mxfp8_gemm(q, s, wq, ws, n, rows=m, bias=b, out=out, residual=out, gate=g, nonfinite=flag)
    gy = om.bf16_round(gate.float().numpy()[None] * y)
    ref = om.bf16_round(res.float().numpy()[rows] + gy)
    check(out, rows, ref, np.abs(gate.float().numpy())[None] * limit + om.bf16_ulp(gy) + om.bf16_ulp(ref))
    assert int(flag.item()) == 0
    # the producer form sums in the same order: the bytes of the separate passes
    for act, fn in ((None, vm.launch_quantize), ("gelu_tanh", vm.launch_gelu_quantize)):
        fq, fs = vm.mxfp8_gemm_act_quantize(q, s, wq, ws, n, rows=m, bias=b, act=act)
        rq, rs = fn(plain)[:2]
        assert torch.equal(fq, rq) and torch.equal(fs, rs), act


@pytest.mark.parametrize("m,f,k,large_rows", [(77, 1280, 1152, 0), (1560, 2560, 1536, 0),
                                              (3330, 2816, 1024, 0), (260, 200, 128, 0),
                                              (2040, 4096, 1280, 2048), (4097, 4000, 1024, 4224),
                                              (4097, 4000, 2048, 4096)])
def test_stream_swiglu_matches_separate_passes(device, m, f, k, large_rows):
    """The SwiGLU producer against the same interleaved GEMM, regrouped, and the stand-alone
    producer: the same bytes, from the stream kernel, the large kernel (whole tiles, and ragged in
    rows and columns) and both in one call."""
    assert_plan(m, -(-f // 128) * 256, k, 3, large_rows, 0 if large_rows >= m else 256)
    g = torch.Generator().manual_seed(m + f)
    x = (torch.randn(m, k, generator=g) * 2).to(torch.bfloat16).to(device)
    w, b = vm.interleave_swiglu((torch.randn(2 * f, k, generator=g) * 0.05).to(torch.bfloat16),
                                torch.randn(2 * f, generator=g).to(torch.bfloat16))
    q, s = vm.quantize_activation(x)
    wq, ws = vm.quantize_activation(w.to(device))
    fq, fs = vm.mxfp8_gemm_act_quantize(q, s, wq, ws, f, rows=m, bias=b.to(device), act="swiglu")
    fp = wq.shape[0] // 2
    y = vm.mxfp8_gemm(q, s, wq, ws, 2 * fp, rows=m, bias=b.to(device))
    y = y.view(m, fp // 128, 2, 128).transpose(1, 2).reshape(m, 2, fp)[:, :, :f].reshape(m, 2 * f)
    rq, rs, _ = vm.launch_swiglu_quantize(y)
    assert torch.equal(fq, rq) and torch.equal(fs, rs)


def test_stream_gemm_flags_nonfinite(device):
    """An inf in the last row reaches the flag from the stream kernel, the large kernel and the
    rows below it; as no row of the output it does not."""
    for m, n, k, large_rows, tile_cols in ((77, 1280, 1152, 0, 128), (512, 5120, 256, 0, 128),
                                           (2040, 8192, 1280, 2048, 0), (2177, 8192, 2304, 2048, 128)):
        assert_plan(m, n, k, 0, large_rows, tile_cols)
        x = torch.ones(m, k, dtype=torch.bfloat16)
        x[m - 1] = 3e38
        q, s = vm.quantize_activation(x.to(device))
        wq, ws = vm.quantize_activation(torch.ones(n, k, dtype=torch.bfloat16, device=device))
        flag = torch.zeros(1, dtype=torch.int32, device=device)
        vm.mxfp8_gemm(q, s, wq, ws, n, rows=m, nonfinite=flag)
        assert int(flag.item()) != 0
        flag.zero_()
        vm.mxfp8_gemm(q, s, wq, ws, n, rows=m - 1, nonfinite=flag)   # that row is no output now
        assert int(flag.item()) == 0


@pytest.mark.parametrize("m,n,k,large_rows,tile_cols", [(77, 1280, 1152, 0, 128), (2040, 8192, 1280, 2048, 0),
                                                        (2177, 8192, 2304, 2048, 128)])
def test_padding_rows_of_the_operand_do_not_matter(device, m, n, k, large_rows, tile_cols):
    """Codes and scales that are NaN in the operand's rows past M (empty_activation leaves them as the
    memory was with zero_padding=False) reach neither the output nor the non-finite flag."""
    assert_plan(m, n, k, 1, large_rows, tile_cols)
    g = torch.Generator().manual_seed(m)
    q, s = vm.quantize_activation(torch.randn(m, k, generator=g).to(torch.bfloat16).to(device))
    wq, ws = vm.quantize_activation((torch.randn(n, k, generator=g) * 0.05).to(torch.bfloat16).to(device))
    res = torch.randn(m, n, generator=g).to(torch.bfloat16).to(device)
    dirty, scales = q.clone(), om.unswizzle(s.cpu().numpy(), *q.shape)
    dirty[m:] = 0xff
    scales[m:] = 0xff
    ds = torch.from_numpy(om.swizzle(scales)).to(device)
    flag = torch.zeros(1, dtype=torch.int32, device=device)
    for r in (None, res):
        ref = vm.mxfp8_gemm(q, s, wq, ws, n, rows=m, residual=r)
        assert torch.equal(vm.mxfp8_gemm(dirty, ds, wq, ws, n, rows=m, residual=r, nonfinite=flag), ref)
    assert int(flag.item()) == 0


def wide(rows, k, g):
    """Normal values whose 32-column MXFP8 blocks lie up to 2^10 apart: their products' sums are far
    from exact in fp32, so another order of them shows."""
    scale = 2.0 ** torch.randint(-5, 6, (rows, k // 32, 1), generator=g)
    return (torch.randn(rows, k // 32, 32, generator=g) * scale).reshape(rows, k).to(torch.bfloat16)


@pytest.mark.parametrize("k", [256, 5120])
def test_rows_do_not_depend_on_the_call(device, k):
    """A row's output is the same bytes whatever number of rows the call has, and whichever kernels
    that number takes: every kernel sums an output over K in one sequence. 1560 and 2177 rows leave
    tiles over after whole rounds of the CUs; 77 and 300 have fewer tiles than CUs."""
    n, rows = 5120, 3330
    g = torch.Generator().manual_seed(k)
    x = wide(rows, k, g).to(device)
    wq, ws = vm.quantize_activation((wide(n, k, g) * 0.05).to(device))
    b = torch.randn(n, generator=g).to(torch.bfloat16).to(device)
    # the general tile kernel: rows of the output that 16-byte accesses do not cover
    store = torch.empty(rows, n + 1, dtype=torch.bfloat16, device=device)
    q, s = vm.quantize_activation(x)
    ref = vm.mxfp8_gemm(q, s, wq, ws, n, rows=rows, bias=b, out=store[:, :n])
    rq = vm.launch_quantize(ref.contiguous())[0]
    for m in (1, 77, 300, 512, 960, 1560, 2177, rows):
        q, s = vm.quantize_activation(x[:m])
        got = vm.mxfp8_gemm(q, s, wq, ws, n, rows=m, bias=b)
        assert torch.equal(got, ref[:m]), m
        pq, _ = vm.mxfp8_gemm_act_quantize(q, s, wq, ws, n, rows=m, bias=b, act=None)
        assert torch.equal(pq[:m], rq[:m]), m


@pytest.mark.parametrize("m,n", [(77, 100), (77, 5119), (1560, 5119)])
def test_producer_matches_separate_passes_at_odd_widths(device, m, n):
    """A width that 16-byte accesses do not cover takes the general kernel for bf16 output and the
    planned ones for the producer: the same bytes, also over many K steps."""
    k = 5120
    g = torch.Generator().manual_seed(m + n)
    q, s = vm.quantize_activation(wide(m, k, g).to(device))
    wq, ws = vm.quantize_activation((wide(n, k, g) * 0.05).to(device))
    y = vm.mxfp8_gemm(q, s, wq, ws, n, rows=m)
    for act, fn in ((None, vm.launch_quantize), ("gelu_tanh", vm.launch_gelu_quantize)):
        fq, fs = vm.mxfp8_gemm_act_quantize(q, s, wq, ws, n, rows=m, act=act)
        rq, rs = fn(y)[:2]
        assert torch.equal(fq, rq) and torch.equal(fs, rs), act


def test_workspace_forms_match(device):
    """The entry points with a workspace run the same launches as those without."""
    m, n, k = 77, 1280, 1152
    g = torch.Generator().manual_seed(9)
    q, s = vm.quantize_activation(wide(m, k, g).to(device))
    wq, ws = vm.quantize_activation(wide(n, k, g).to(device))
    size = ctypes.c_int64(-1)
    _lib.call("vdn_mxfp8_gemm_workspace", q.shape[0], wq.shape[0], k, 0, ctypes.byref(size))
    assert size.value == 0
    work = torch.empty(1 << 20, dtype=torch.uint8, device=device)
    ref = vm.mxfp8_gemm(q, s, wq, ws, n, rows=m)
    rq, rs = vm.mxfp8_gemm_act_quantize(q, s, wq, ws, n, rows=m)
    out, cq, cs = torch.zeros_like(ref), torch.zeros_like(rq), torch.zeros_like(rs)
    head = (q.data_ptr(), s.data_ptr(), q.shape[0], wq.data_ptr(), ws.data_ptr(), wq.shape[0], k, None)
    for space in ((work.data_ptr(), work.numel()), (None, 0)):
        _lib.call("vdn_mxfp8_gemm_ws", *head, None, 0, None, 0, None, out.data_ptr(), m, n, n, None,
                  *space, _lib.stream(device))
        _lib.call("vdn_mxfp8_gemm_act_quantize_ws", *head, 1, cq.data_ptr(), cs.data_ptr(), m, n, None,
                  *space, _lib.stream(device))
        assert torch.equal(out, ref) and torch.equal(cq, rq) and torch.equal(cs, rs)
    with pytest.raises(RuntimeError, match="alignment"):
        _lib.call("vdn_mxfp8_gemm_ws", *head, None, 0, None, 0, None, out.data_ptr(), m, n, n, None,
                  work.data_ptr() + 4, 1024, _lib.stream(device))
