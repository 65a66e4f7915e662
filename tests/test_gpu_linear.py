"""GPU parity of the attention projections on the MFMA kernels (linear.py).

rv_linear_fwd / rv_linear_dx / rv_linear_dw against the fp64 contraction of
the same fp16 operands, within the fp32-accumulation bound of
tests/gemm_bounds.py; FusedLinear against autocast's F.linear (forward and
both gradients); enable_linear leaves unsupported calls on F.linear.
"""
from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from gemm_bounds import TILE_WIDTHS, rel_l2, within_gemm_bound
from reversability_amd import mlp
from reversability_amd._hip import RV_F16, RV_F32, _check, _stream, library
from reversability_amd.linear import FusedLinear, enable_linear, linear, supported

pytestmark = pytest.mark.gpu

# (rows, in, out): configs[3] qkv / proj over the batch, a ragged row count,
# configs[4] qkv / proj
SHAPES = [(16896, 256, 768), (16896, 256, 256), (1000, 256, 768), (32768, 1024, 3072),
          (32768, 1024, 1024)]


def _data(rows, in_f, out_f, dev, seed=7):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(rows, in_f, generator=g).half().to(dev)
    w = (0.02 * torch.randn(out_f, in_f, generator=g)).to(dev)
    dy = torch.randn(rows, out_f, generator=g).half().to(dev)
    return x, w, dy


@pytest.mark.parametrize("rows,in_f,out_f", SHAPES)
def test_linear_kernels_vs_fp64(cuda_device, rows, in_f, out_f):
    x, w, dy = _data(rows, in_f, out_f, cuda_device)
    w16 = mlp.cast_f16(w)
    lib = library()
    y = torch.empty(rows, out_f, device=cuda_device, dtype=torch.float16)
    _check(lib.rv_linear_fwd(x.data_ptr(), in_f, w16.data_ptr(), rows, in_f, out_f, y.data_ptr(),
                             _stream(x)), "fwd")
    assert within_gemm_bound(y, x, w16, in_f)
    for dt, code in ((torch.float32, RV_F32), (torch.float16, RV_F16)):
        dx = torch.empty(rows, in_f, device=cuda_device, dtype=dt)
        _check(lib.rv_linear_dx(dy.data_ptr(), w16.data_ptr(), rows, in_f, out_f, dx.data_ptr(),
                                code, _stream(x)), "dx")
        assert within_gemm_bound(dx, dy, w16, out_f, transpose_b=False)
        if dt == torch.float32:
            assert torch.equal(dx, dx.half().float())
    nbytes = lib.rv_linear_dw_workspace_bytes(rows, in_f, out_f)
    ws = torch.empty(max(nbytes, 4) // 4, device=cuda_device)
    dw = torch.empty(out_f, in_f, device=cuda_device)
    _check(lib.rv_linear_dw(dy.data_ptr(), x.data_ptr(), in_f, rows, in_f, out_f, dw.data_ptr(), 0,
                            ws.data_ptr(), nbytes, _stream(x)), "dw")
    assert torch.equal(dw, dw.half().float())
    assert within_gemm_bound(dw, dy.t(), x.t(), rows)
    first = dw.clone()
    _check(lib.rv_linear_dw(dy.data_ptr(), x.data_ptr(), in_f, rows, in_f, out_f, dw.data_ptr(), 1,
                            ws.data_ptr(), nbytes, _stream(x)), "dw acc")
    assert torch.equal(dw, first + first)


@pytest.mark.parametrize("xdtype", [torch.float32, torch.float16])
def test_fused_linear_matches_autocast_linear(cuda_device, xdtype):
    g = torch.Generator().manual_seed(11)
    x = torch.randn(33, 512, 256, generator=g).to(cuda_device).to(xdtype)
    w = (0.02 * torch.randn(768, 256, generator=g)).to(cuda_device)
    gy = torch.randn(33, 512, 768, generator=g).half().to(cuda_device)
    xa, wa = x.clone().requires_grad_(True), w.clone().requires_grad_(True)
    xb, wb = x.clone().requires_grad_(True), w.clone().requires_grad_(True)
    with torch.autocast("cuda", dtype=torch.float16):
        assert supported(xb, wb, None)
        ya = F.linear(xa, wa)
        yb = FusedLinear.apply(xb, wb)
    assert ya.dtype == yb.dtype == torch.float16 and yb.shape == ya.shape
    ya.backward(gy)
    yb.backward(gy)
    assert xb.grad.dtype == xdtype and wb.grad.dtype == torch.float32
    assert rel_l2(yb, ya) < 1e-3
    assert rel_l2(xb.grad, xa.grad) < 1e-3
    assert rel_l2(wb.grad, wa.grad) < 1e-3


def test_enable_linear_falls_back_outside_fp16_autocast(cuda_device):
    from reversability_amd import build_model
    torch.manual_seed(0)
    model = build_model({"model": {"vocab_size": 97, "max_sequence_length": 32, "n_layers": 1,
                                   "n_heads": 8, "d_model": 256, "d_ff": 1024},
                         "method": "midpoint"}).to(cuda_device)
    enable_linear(model)
    x = torch.randn(2, 32, 256, device=cuda_device)
    layer = model.blocks[0].attn.qkv
    # no autocast: plain fp32 F.linear
    assert torch.equal(layer(x), F.linear(x, layer.weight))
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert not supported(x, layer.weight, None)
        assert layer(x).dtype == torch.bfloat16
    with torch.autocast("cuda", dtype=torch.float16):
        assert supported(x, layer.weight, None)
        assert linear(x, layer.weight).dtype == torch.float16


@pytest.mark.parametrize("rows,in_f,out_f", [(1, 2048, 128), (51, 4096, 256), (65, 8192, 128),
                                             (512, 4096, 1024), (500, 4224, 1152)])
def test_split_reduction(cuda_device, rows, in_f, out_f):
    """Products with few output tiles and a long reduction are split over it:
    the fp64 bound for the forward and the fp16 and fp32 input gradients,
    identical bits on every tile shape, and a workspace that is too small is
    refused."""
    from reversability_amd._hip import RV_F16, RV_F32, _stream, library
    lib = library()
    g = torch.Generator().manual_seed(23)
    x = torch.randn(rows, in_f, generator=g).half().to(cuda_device)
    w = (0.02 * torch.randn(out_f, in_f, generator=g)).half().to(cuda_device)
    wt = w.t().contiguous()  # [in_f, out_f]: dx of a layer with out = in_f, in = out_f
    need = lib.rv_linear_splitk_workspace_bytes(rows, out_f, in_f)
    assert need > 0 and need % (4 * rows * out_f) == 0
    ws = torch.empty(need // 4, device=cuda_device)
    st = _stream(x)
    first = None
    try:
        for shape in range(-1, lib.rv_gemm_num_shapes()):
            assert lib.rv_gemm_force_shape(shape) == 0
            y, d16 = (torch.empty(rows, out_f, device=cuda_device, dtype=torch.float16)
                      for _ in range(2))
            d32 = torch.empty(rows, out_f, device=cuda_device)
            args = (ws.data_ptr(), need, st)
            codes = [lib.rv_linear_fwd_ws(x.data_ptr(), in_f, w.data_ptr(), rows, in_f, out_f,
                                          y.data_ptr(), *args)]
            for dx, code in ((d16, RV_F16), (d32, RV_F32)):
                codes.append(lib.rv_linear_dx_ws(x.data_ptr(), wt.data_ptr(), rows, out_f, in_f,
                                                 dx.data_ptr(), code, *args))
            if shape >= 0 and out_f % TILE_WIDTHS[shape]:
                assert codes == [3, 3, 3], shape
                continue
            assert codes == [0, 0, 0], shape
            if first is None:
                first = (y, d16, d32)
                assert within_gemm_bound(y, x, w, in_f)
                assert within_gemm_bound(d16, x, w, in_f)
                assert torch.equal(d32, d16.float())
            else:
                assert all(torch.equal(a, b) for a, b in zip(first, (y, d16, d32))), shape
    finally:
        lib.rv_gemm_force_shape(-1)
    assert lib.rv_linear_fwd_ws(x.data_ptr(), in_f, w.data_ptr(), rows, in_f, out_f,
                                first[0].data_ptr(), ws.data_ptr(), need - 1, st) != 0


@pytest.mark.parametrize("xdtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("batch,seq,heads,hd", [(1, 1, 4, 32), (3, 17, 8, 32), (2, 130, 4, 64),
                                                (1, 257, 3, 128), (5, 96, 16, 64)])
def test_attention_layer_matches_its_parts(cuda_device, batch, seq, heads, hd, xdtype):
    """The one-node attention layer against the three Functions it stands for
    (a forward hook on a projection keeps the parts): the same output and
    input-gradient bits, weight gradients within 2e-3 (their rows are summed
    in another order, as a lone layer's are), frozen weights, and the same recorded paths."""
    from reversability_amd import paths
    from reversability_amd.attention import AttentionLayer, enable_attention
    from reversability_amd.model import BaselineLM, ModelConfig
    d = heads * hd
    torch.manual_seed(3)
    model = BaselineLM(ModelConfig(vocab_size=64, max_sequence_length=seq, n_layers=1,
                                   n_heads=heads, d_model=d, d_ff=d)).to(cuda_device)
    enable_linear(model)
    enable_attention(model)
    attn = model.blocks[0].attn
    g = torch.Generator().manual_seed(7)
    x = torch.randn(batch, seq, d, generator=g).to(cuda_device, xdtype).requires_grad_(True)
    dy = torch.randn(batch, seq, d, generator=g).half().to(cuda_device)
    leaves = (x, attn.qkv.weight, attn.proj.weight)

    def once(wanted=leaves):
        paths.reset()
        with torch.autocast("cuda", dtype=torch.float16):
            y = attn(x)
        node = type(y.grad_fn).__name__
        return y, torch.autograd.grad(y, wanted, dy), node, paths.report()

    y, grads, node, report = once()
    assert node == AttentionLayer.__name__ + "Backward"
    frozen = once((x,))[1]
    handle = attn.proj.register_forward_hook(lambda *a: None)
    y_parts, grads_parts, node_parts, report_parts = once()
    handle.remove()
    assert node_parts != node and report == report_parts
    assert torch.equal(y, y_parts) and torch.equal(grads[0], grads_parts[0])
    assert torch.equal(frozen[0], grads[0])
    for a, b in zip(grads[1:], grads_parts[1:]):
        assert rel_l2(a, b) < 2e-3
    attn.qkv.weight.requires_grad_(False)
    partial = once((x, attn.proj.weight))[1]
    assert torch.equal(partial[0], grads[0]) and rel_l2(partial[1], grads[2]) < 2e-3
    x.requires_grad_(False)  # the output projection alone: no attention backward
    assert torch.equal(once((attn.proj.weight,))[1][0], partial[1])
    attn.qkv.weight.requires_grad_(True)
    attn.proj.weight.requires_grad_(False)
    assert rel_l2(once((attn.qkv.weight,))[1][0], grads[1]) < 2e-3
