"""GPU parity of the fused cross-entropy (rv_ce_fwd / rv_ce_bwd).

* The reference's own test (tests/test_kernels.py:19-37): 17 x 50257 logits
  with labels at both vocabulary ends, a tile edge and an ignored row, against
  eager F.cross_entropy (fp16 under autocast, and fp32), scaled backward;
  rtol = atol = 2e-3 on the loss, gradient relative L2 < 2e-2 (fp16) /
  2e-5 (fp32), the ignored row's gradient exactly zero.
* Against the CPU oracle: row max bit-exact; log-sum-exp within fp32
  summation-order error; per-row loss within one fp16 ulp (the rounding of
  the log-probability can flip when the fp32 log-sum-exp differs in its last
  bit); the backward, given the kernel's own row statistics, within one ulp
  on every element and identical on > 99%.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch
import torch.nn.functional as F

import oracle
from reversability_amd.kernels import TiledCrossEntropy, cross_entropy_sum
from reversability_amd._hip import ops

pytestmark = pytest.mark.gpu

LABELS17 = [0, 1023, 1024, 50256, -100] + list(range(12))


def ulp16(v):
    return np.spacing(np.abs(np.asarray(v, np.float64)).astype(np.float16)).astype(np.float64)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_reference_full_vocabulary_tail_mask_and_scaled_backward(cuda_device, dtype):
    torch.manual_seed(41)
    a = torch.randn(17, 50257, device=cuda_device, dtype=dtype, requires_grad=True)
    b = a.detach().clone().requires_grad_(True)
    y = torch.tensor(LABELS17, device=cuda_device)
    with torch.autocast("cuda", enabled=dtype == torch.float16, dtype=torch.float16):
        expected = F.cross_entropy(a, y, reduction="sum", ignore_index=-100)
    actual = cross_entropy_sum(b, y)
    (expected * .03125).backward()
    (actual * .03125).backward()
    torch.testing.assert_close(actual, expected.float(), rtol=.002, atol=.002)
    relative = (a.grad.float() - b.grad.float()).norm() / a.grad.float().norm()
    assert relative < (.02 if dtype == torch.float16 else 2e-5)
    assert torch.count_nonzero(b.grad[4]) == 0


@pytest.mark.parametrize("rows,cols,dtype", [(1024, 50257, torch.float16), (17, 50257, torch.float32),
                                             (5, 7, torch.float16), (33, 1000, torch.float16),
                                             (9, 4096, torch.float32)])
def test_matches_oracle(cuda_device, rows, cols, dtype):
    g = torch.Generator().manual_seed(rows * 7 + cols)
    x = (3 * torch.randn(rows, cols, generator=g)).to(dtype)
    y = torch.randint(0, cols, (rows,), generator=g)
    y[::5] = -100
    xd, yd = x.to(cuda_device), y.to(cuda_device)
    rmax, rlse, loss = ops.ce_fwd(xd, yd, -100)
    omax, olse, oloss = oracle.ce_fwd(x.numpy(), y.numpy())
    assert np.array_equal(rmax.cpu().numpy(), omax)
    assert np.all(np.abs(rlse.cpu().numpy() - olse) <= 2e-6 * np.abs(olse) + 2e-6)
    lg = loss.cpu().numpy()
    if dtype == torch.float16:
        assert np.all(np.abs(lg - oloss) <= ulp16(oloss))
        assert np.mean(lg == oloss) > 0.95
    else:
        assert np.all(np.abs(lg - oloss) <= 1e-5 * np.abs(oloss) + 1e-6)
    grad = torch.tensor([0.75], device=cuda_device)
    dx = ops.ce_bwd(xd, yd, rmax, rlse, grad, -100).cpu()
    odx = oracle.ce_bwd(x.numpy(), y.numpy(), rmax.cpu().numpy(), rlse.cpu().numpy(), 0.75)
    dg, do = dx.numpy().astype(np.float64), odx.astype(np.float64)
    if dtype == torch.float16:
        assert np.all(np.abs(dg - do) <= ulp16(do) + 1e-12)
        assert np.mean(dg == do) > 0.99
    else:
        assert np.all(np.abs(dg - do) <= 1e-5 * np.abs(do) + 1e-9)
    assert torch.count_nonzero(dx[::5]) == 0


def test_deterministic_and_bad_labels(cuda_device):
    x = torch.randn(8, 50257, device=cuda_device).half()
    y = torch.tensor([1, 2, 50257, -1, 5, 6, 7, -100], device=cuda_device)
    a = ops.ce_fwd(x, y, -100)
    b = ops.ce_fwd(x, y, -100)
    # bitwise identical, NaN rows included
    assert all(torch.equal(torch.isnan(u), torch.isnan(v)) and torch.equal(u.nan_to_num(), v.nan_to_num())
               for u, v in zip(a, b))
    loss = a[2].cpu()
    assert torch.isnan(loss[2]) and torch.isnan(loss[3]) and torch.isfinite(loss[[0, 1, 4, 5, 6]]).all()
    assert loss[7] == 0


def test_rejects_cpu_and_bad_inputs(cuda_device):
    with pytest.raises(ValueError, match="CUDA"):
        cross_entropy_sum(torch.zeros(3, 31), torch.tensor([0, 1, -100]))
    x = torch.zeros(3, 31, device=cuda_device, dtype=torch.float16)
    with pytest.raises(ValueError, match="int64"):
        TiledCrossEntropy.apply(x, torch.tensor([0, 1, 2], device=cuda_device, dtype=torch.int32))
    with pytest.raises(ValueError, match="Contiguous"):
        TiledCrossEntropy.apply(x.t(), torch.tensor([0, 1, 2], device=cuda_device))


@pytest.mark.parametrize("rows,d,vocab", [(1000, 256, 50257), (333, 128, 1001), (64, 256, 64),
                                           (64, 64, 70001), (64, 128, 70001),
                                           # the routes of head_routes (own logits, own gradients)
                                           (5100, 1024, 4001),   # no, yes
                                           (8200, 384, 1001)])   # yes, no
def test_tied_head_ce_matches_autograd(cuda_device, rows, d, vocab):
    """The padded-stride head + fused CE (forward and backward in one call;
    two passes above 65536 columns) against autograd of autocast F.linear +
    cross_entropy_sum on the same fp16 operands: the same loss and gradients
    up to the GEMMs' fp32 accumulation order (the MFMA kernels', or the library's
    at a padded row stride)."""
    from reversability_amd.kernels import padded_head, tied_head_ce
    g = torch.Generator().manual_seed(5)
    x16 = torch.randn(rows, d, generator=g).half().to(cuda_device)
    w = (0.05 * torch.randn(vocab, d, generator=g)).to(cuda_device)
    labels = torch.randint(0, vocab, (rows,), generator=g).to(cuda_device)
    labels[::7] = -100
    grad = torch.tensor([0.37], device=cuda_device)
    head16 = padded_head(w)
    assert head16.shape[0] % 64 == 0 and torch.equal(head16[vocab:], torch.zeros_like(head16[vocab:]))
    # memory that the call's buffers take over (the logits' pad columns among them)
    used = [torch.full((rows, head16.shape[0]), float("nan"), device=cuda_device,
                       dtype=torch.float16) for _ in range(2)]
    del used
    loss, dx16, dw16 = tied_head_ce(x16, head16, vocab, labels, grad)
    xr = x16.clone().requires_grad_(True)
    hr = w.half().requires_grad_(True)
    ref = cross_entropy_sum(torch.nn.functional.linear(xr, hr), labels)
    (ref * 0.37).backward()
    ref = float(ref.detach())
    assert abs(float(loss) - ref) <= 1e-3 * abs(ref)
    assert dx16.shape == (rows, d) and dw16.shape == (vocab, d) and dw16.is_contiguous()
    for got, want in ((dx16, xr.grad), (dw16, hr.grad)):
        assert got.dtype == torch.float16
        rel = float((got.float() - want.float()).norm() / want.float().norm())
        assert rel < 2e-3, rel


def _fused_vs_two_pass(lib, flat, offset, ld, cols, y, grad, in_place):
    """rv_ce_fused on the rows of stride ld starting at flat[offset] (first cols
    used) against rv_ce_fwd followed by rv_ce_bwd on a copy; returns both
    (row max, lse, loss, dlogits).  Copies keep flat's address modulo 16."""
    from reversability_amd._hip import RV_F16, _stream
    rows = y.numel()
    dev = flat.device
    outs = []
    for fused in (True, False):
        xs = flat.clone()
        x = xs[offset:offset + rows * ld]
        st = [torch.full((rows,), 7.0, device=dev) for _ in range(3)]
        d = x if (fused and in_place) else torch.full_like(xs, 3.0)[offset:offset + rows * ld]
        assert (x.data_ptr() - d.data_ptr()) % 16 == 0
        ptrs = [t.data_ptr() for t in st]
        if fused:
            rc = lib.rv_ce_fused(x.data_ptr(), RV_F16, ld, y.data_ptr(), rows, cols, -100,
                                 grad.data_ptr(), *ptrs, d.data_ptr(), _stream(xs))
            assert rc == 0
        else:
            assert lib.rv_ce_fwd(x.data_ptr(), RV_F16, ld, y.data_ptr(), rows, cols, -100,
                                 *ptrs, _stream(xs)) == 0
            assert lib.rv_ce_bwd(x.data_ptr(), RV_F16, ld, y.data_ptr(), ptrs[0], ptrs[1],
                                 grad.data_ptr(), rows, cols, -100, d.data_ptr(),
                                 _stream(xs)) == 0
        torch.cuda.synchronize()
        outs.append((*st, d.view(rows, ld)))
    return outs


def _same_bits(a, b):
    return torch.equal(a.view(torch.int16) if a.dtype == torch.float16 else a.view(torch.int32),
                       b.view(torch.int16) if b.dtype == torch.float16 else b.view(torch.int32))


@pytest.mark.parametrize("rows,cols,ld,offset", [
    (64, 50257, 50304, 0),     # the tied head's padded stride
    (37, 50257, 50257, 0),     # odd stride: every row has a scalar head and tail
    (19, 65536, 65536, 0),     # widest row the registers hold
    (11, 65535, 65536, 3),     # misaligned base, 16 vectors per thread
    (23, 2048, 2051, 5),
    (9, 7, 8, 1),              # no vector part
    (5, 1, 1, 0),
    (256, 3000, 3072, 0),
])
@pytest.mark.parametrize("in_place", [False, True])
def test_fused_matches_two_pass_bitwise(cuda_device, rows, cols, ld, offset, in_place):
    """rv_ce_fused = rv_ce_fwd then rv_ce_bwd, bit for bit (row max, lse,
    loss, every written dlogits element incl. ignored and bad-label rows);
    the padding past cols is left as it was."""
    from reversability_amd._hip import library
    g = torch.Generator().manual_seed(rows + cols)
    flat = (4 * torch.randn(rows * ld + offset, generator=g)).half().to(cuda_device)
    y = torch.randint(0, cols, (rows,), generator=g)
    y[::4] = -100
    if rows > 5:
        y[1], y[2], y[3] = cols - 1, cols, -7   # last column; two bad labels
    y = y.to(cuda_device)
    if rows > 5 and cols > 64:
        # a row spanning the fp16 range: exp(logp) underflows (zero-signed gradients)
        flat[offset + 5 * ld:offset + 5 * ld + cols] = torch.linspace(
            -60000.0, 8.0, cols, device=cuda_device).half()
    grad = torch.tensor([0.3125], device=cuda_device)
    (fm, fl, floss, fd), (tm, tl, tloss, td) = _fused_vs_two_pass(library(), flat, offset, ld, cols,
                                                                   y, grad, in_place)
    assert _same_bits(fm, tm) and _same_bits(fl, tl) and _same_bits(floss, tloss)
    assert _same_bits(fd[:, :cols], td[:, :cols])
    if ld > cols and not in_place:
        assert bool((fd[:, cols:] == 3.0).all())
    if rows > 5:
        assert torch.isnan(floss[2]) and torch.isnan(floss[3])
        assert torch.isnan(fd[2, :cols].float()).all()
    assert torch.count_nonzero(fd[::4, :cols]) == 0


def test_fused_matches_oracle_and_rejects_wide_rows(cuda_device):
    """Against the CPU oracle (loss within one fp16 ulp, dlogits within one ulp
    given the kernel's own statistics), and RV_ERR_UNSUPPORTED for fp32 and
    rows wider than 65536 (the caller takes the two-pass kernels)."""
    from reversability_amd._hip import RV_F16, RV_F32, _stream, library
    lib = library()
    rows, cols = 200, 50257
    g = torch.Generator().manual_seed(9)
    x = (3 * torch.randn(rows, cols, generator=g)).half()
    y = torch.randint(0, cols, (rows,), generator=g)
    y[::5] = -100
    xd, yd = x.to(cuda_device), y.to(cuda_device)
    grad = torch.tensor([0.75], device=cuda_device)
    rmax, rlse, loss = (torch.empty(rows, device=cuda_device) for _ in range(3))
    dx = torch.empty_like(xd)
    assert lib.rv_ce_fused(xd.data_ptr(), RV_F16, cols, yd.data_ptr(), rows, cols, -100,
                           grad.data_ptr(), rmax.data_ptr(), rlse.data_ptr(), loss.data_ptr(),
                           dx.data_ptr(), _stream(xd)) == 0
    omax, olse, oloss = oracle.ce_fwd(x.numpy(), y.numpy())
    assert np.array_equal(rmax.cpu().numpy(), omax)
    lg = loss.cpu().numpy()
    assert np.all(np.abs(lg - oloss) <= ulp16(oloss))
    odx = oracle.ce_bwd(x.numpy(), y.numpy(), rmax.cpu().numpy(), rlse.cpu().numpy(), 0.75)
    dg, do = dx.cpu().numpy().astype(np.float64), odx.astype(np.float64)
    assert np.all(np.abs(dg - do) <= ulp16(do) + 1e-12)
    assert np.mean(dg == do) > 0.99
    RV_ERR_UNSUPPORTED = 3  # include/reversibility_hip.h
    wide = torch.zeros(2, 65544, device=cuda_device, dtype=torch.float16)
    y2 = torch.zeros(2, device=cuda_device, dtype=torch.int64)
    args = (y2.data_ptr(), 2, 65544, -100, grad.data_ptr(), rmax.data_ptr(), rlse.data_ptr(),
            loss.data_ptr(), wide.data_ptr(), _stream(wide))
    assert lib.rv_ce_fused(wide.data_ptr(), RV_F16, 65544, *args) == RV_ERR_UNSUPPORTED
    assert lib.rv_ce_fused(wide.data_ptr(), RV_F32, 65544, *args) == RV_ERR_UNSUPPORTED


@pytest.mark.parametrize("rows,d,vocab", [(1, 128, 161), (65, 256, 1001), (300, 384, 192),
                                           (513, 128, 7000), (700, 256, 9999)])
def test_head_products(cuda_device, rows, d, vocab):
    """The head's three GEMMs at vocabularies whose padded width is not a
    multiple of the tiles: the fp64 bound, identical bits on every tile shape,
    pad columns zero also for a row of infinities, dW as fp16, widened, and
    accumulated, from one workspace."""
    from gemm_bounds import TILE_WIDTHS, within_gemm_bound
    from reversability_amd._hip import RV_F16, RV_F32, _stream, library
    lib = library()
    assert lib.rv_gemm_num_shapes() == len(TILE_WIDTHS)
    padded = -(-vocab // 64) * 64
    g = torch.Generator().manual_seed(19)
    x = torch.randn(rows, d, generator=g).half().to(cuda_device)
    head = torch.zeros(padded, d)
    head[:vocab] = 0.05 * torch.randn(vocab, d, generator=g)
    head = head.half().to(cuda_device)
    grad = torch.zeros(rows, padded)
    grad[:, :vocab] = 1e-2 * torch.randn(rows, vocab, generator=g)
    grad = grad.half().to(cuda_device)
    size = (rows, d, vocab, padded)
    st = _stream(x)
    nbytes = lib.rv_head_workspace_bytes(*size)
    assert nbytes >= 0
    ws = torch.empty(max(nbytes, 16) // 4, device=cuda_device)
    first = None
    try:
        for shape in range(-1, lib.rv_gemm_num_shapes()):
            assert lib.rv_gemm_force_shape(shape) == 0
            logits = torch.full((rows, padded), 3.0, device=cuda_device, dtype=torch.float16)
            dx = torch.empty_like(x)
            assert lib.rv_head_logits(x.data_ptr(), head.data_ptr(), *size, logits.data_ptr(),
                                      st) == 0
            rc = lib.rv_head_dx(grad.data_ptr(), head.data_ptr(), *size, dx.data_ptr(),
                                ws.data_ptr(), nbytes, st)
            fits = shape < 0 or d % TILE_WIDTHS[shape] == 0
            assert rc == (0 if fits else 3), shape
            if not fits:  # refused: only the logits are compared
                dx = first[1]
            if first is None:
                first = (logits, dx)
                assert within_gemm_bound(logits, x, head, d)
                assert within_gemm_bound(dx, grad, head, padded, transpose_b=False)
            assert torch.equal(logits, first[0]) and torch.equal(dx, first[1]), shape
    finally:
        lib.rv_gemm_force_shape(-1)
    dw16 = torch.empty(vocab, d, device=cuda_device, dtype=torch.float16)
    dw32 = torch.empty(vocab, d, device=cuda_device)
    call = lambda out, code, acc: lib.rv_head_dw(
        grad.data_ptr(), x.data_ptr(), *size, out.data_ptr(), code, acc, ws.data_ptr(), nbytes, st)
    assert call(dw16, RV_F16, 0) == 0 and call(dw32, RV_F32, 0) == 0
    assert within_gemm_bound(dw16, grad[:, :vocab].t(), x.t(), rows)
    assert torch.equal(dw32, dw16.float())
    assert call(dw32, RV_F32, 1) == 0
    assert torch.equal(dw32, 2 * dw16.float())
    x[0] = float("inf")
    assert lib.rv_head_logits(x.data_ptr(), head.data_ptr(), *size, logits.data_ptr(), st) == 0
    assert not logits[:, vocab:].any()


def test_head_products_past_32_bit_offsets(cuda_device):
    """A logits matrix above 2 GiB: its last rows' logits and input gradient and
    the whole weight gradient (whose sum runs past the 2 GiB mark) against
    fp32 products of the same operands."""
    from reversability_amd._hip import RV_F32, _stream, library
    lib = library()
    rows, d, vocab, padded = 22000, 128, 50257, 50304
    assert rows * padded * 2 > 1 << 31
    g = torch.Generator(device=cuda_device).manual_seed(3)
    x = torch.randn(rows, d, generator=g, device=cuda_device).half()
    head = torch.zeros(padded, d, device=cuda_device, dtype=torch.float16)
    head[:vocab] = 0.05 * torch.randn(vocab, d, generator=g, device=cuda_device)
    size, st = (rows, d, vocab, padded), _stream(x)
    logits = torch.empty(rows, padded, device=cuda_device, dtype=torch.float16)
    assert lib.rv_head_logits(x.data_ptr(), head.data_ptr(), *size, logits.data_ptr(), st) == 0
    nbytes = lib.rv_head_workspace_bytes(*size)
    ws = torch.empty(max(nbytes, 16) // 4, device=cuda_device)
    dx, dw = torch.empty_like(x), torch.empty(vocab, d, device=cuda_device)
    assert lib.rv_head_dx(logits.data_ptr(), head.data_ptr(), *size, dx.data_ptr(), ws.data_ptr(),
                          nbytes, st) == 0
    assert lib.rv_head_dw(logits.data_ptr(), x.data_ptr(), *size, dw.data_ptr(), RV_F32, 0,
                          ws.data_ptr(), nbytes, st) == 0
    rel = lambda a, b: float((a.float() - b).norm() / b.norm())
    for rows_ in (slice(0, 64), slice(-64, None)):
        assert rel(logits[rows_], x[rows_].float() @ head.float().t()) < 1e-3
        assert rel(dx[rows_], logits[rows_].float() @ head.float()) < 1e-3
    ref = torch.zeros(vocab, d, device=cuda_device)
    for at in range(0, rows, 2000):
        ref += logits[at:at + 2000, :vocab].float().t() @ x[at:at + 2000].float()
    assert rel(dw, ref) < 1e-3


def test_tied_head_ce_refuses_a_wrong_dw_out(cuda_device):
    """The weight gradient's output has to be a contiguous fp32 [vocab, d]; one
    off a 16-byte boundary is taken (torch's products)."""
    from reversability_amd.kernels import padded_head, tied_head_ce
    g = torch.Generator().manual_seed(9)
    x16 = torch.randn(32, 128, generator=g).half().to(cuda_device)
    head16 = padded_head((0.05 * torch.randn(100, 128, generator=g)).to(cuda_device))
    labels = torch.randint(0, 100, (32,), generator=g).to(cuda_device)
    args = (x16, head16, 100, labels, torch.ones(1, device=cuda_device))
    for wrong in (torch.empty(99, 128, device=cuda_device),
                  torch.empty(100, 128, device=cuda_device, dtype=torch.float16),
                  torch.empty(128, 100, device=cuda_device).t(), torch.empty(100, 128)):
        with pytest.raises(ValueError):
            tied_head_ce(*args, dw_out=wrong)
    _, dx, dw = tied_head_ce(*args, dw_out=torch.empty(100, 128, device=cuda_device))
    odd = torch.empty(100 * 128 + 1, device=cuda_device)[1:].view(100, 128)
    _, dx_odd, dw_odd = tied_head_ce(*args, dw_out=odd)
    for a, b in ((dx, dx_odd), (dw, dw_odd)):  # the same products, summed in another order
        assert float((a.float() - b.float()).norm() / a.float().norm()) < 2e-3


@pytest.mark.parametrize("which", ["head16", "labels", "grad", "dx_out"])
def test_tied_head_ce_refuses_other_devices(cuda_device, which):
    """An operand or output in host memory is refused before any kernel gets its pointer."""
    from reversability_amd.kernels import padded_head, tied_head_ce
    g = torch.Generator().manual_seed(9)
    args = {"x16": torch.randn(32, 128, generator=g).half().to(cuda_device),
            "head16": padded_head((0.05 * torch.randn(100, 128, generator=g)).to(cuda_device)),
            "vocab": 100, "labels": torch.randint(0, 100, (32,), generator=g).to(cuda_device),
            "grad": torch.ones(1, device=cuda_device),
            "dx_out": torch.empty(32, 128, device=cuda_device, dtype=torch.float16)}
    _, dx, _ = tied_head_ce(**args)
    assert dx.data_ptr() == args["dx_out"].data_ptr()
    args[which] = args[which].cpu()
    with pytest.raises(ValueError, match="device"):
        tied_head_ce(**args)


@pytest.mark.parametrize("rows,d,vocab", [(48, 128, 1001), (48, 128, 70001), (5100, 1024, 4001)])
def test_head_pad_rows_do_not_matter(cuda_device, rows, d, vocab):
    """Whatever a caller left in the head's pad rows (NaN here), loss and
    gradients are those of zero pad rows, with the one-pass cross-entropy, the
    two-pass one of a wide vocabulary, and torch's product for the logits."""
    from reversability_amd.kernels import padded_head, tied_head_ce
    g = torch.Generator().manual_seed(5)
    x16 = torch.randn(rows, d, generator=g).half().to(cuda_device)
    head16 = padded_head((0.05 * torch.randn(vocab, d, generator=g)).to(cuda_device))
    labels = torch.randint(0, vocab, (rows,), generator=g).to(cuda_device)
    args = (vocab, labels, torch.ones(1, device=cuda_device))
    clean = tied_head_ce(x16, head16, *args)
    head16[vocab:] = float("nan")
    for a, b in zip(clean, tied_head_ce(x16, head16, *args)):
        assert torch.equal(a, b)


def test_head_first_call_does_not_wait(cuda_device):
    """The head's products take their tile shapes from the sizes: a call at a row
    count that no call had before times nothing, so it returns while earlier
    work of the stream still runs."""
    from reversability_amd.kernels import padded_head, tied_head_ce
    g = torch.Generator().manual_seed(9)
    head16 = padded_head((0.05 * torch.randn(1001, 256, generator=g)).to(cuda_device))
    grad = torch.ones(1, device=cuda_device)
    data = [(torch.randn(rows, 256, generator=g).half().to(cuda_device),
             torch.randint(0, 1001, (rows,), generator=g).to(cuda_device))
            for rows in (1237, 1239)]
    for i, (x16, labels) in enumerate(data):  # the first one loads the kernels
        torch.cuda.synchronize()
        torch.cuda._sleep(20_000_000)
        slept = torch.cuda.Event()
        slept.record()
        tied_head_ce(x16, head16, 1001, labels, grad)
        busy = not slept.query()
        torch.cuda.synchronize()
        assert busy or i == 0


def test_tied_head_records_the_sides_taken(cuda_device):
    """The record follows the branch, operands' alignment included."""
    from reversability_amd import paths
    from reversability_amd.kernels import padded_head, tied_head_ce

    def record(rows, d, vocab, **out):
        x16 = torch.zeros(rows, d, device=cuda_device, dtype=torch.float16)
        head16 = padded_head(torch.zeros(vocab, d, device=cuda_device))
        labels = torch.zeros(rows, device=cuda_device, dtype=torch.int64)
        paths.reset()
        tied_head_ce(x16, head16, vocab, labels, torch.ones(1, device=cuda_device), **out)
        return list(paths.report()["tied_head"])

    assert record(32, 128, 100) == ["fused-ce+mfma"]
    assert record(32, 64, 100) == ["fused-ce+hipblaslt"]
    assert record(5100, 1024, 4001) == ["fused-ce+hipblaslt/mfma"]
    off = torch.empty(100 * 128 + 1, device=cuda_device)[1:].view(100, 128)
    assert record(32, 128, 100, dw_out=off) == ["fused-ce+mfma/hipblaslt"]


@pytest.mark.parametrize("offset", [0, 1])  # floats: the kernels' route, and torch's off 16 bytes
def test_tied_head_ce_accumulates_over_chunks(cuda_device, offset):
    """Two chunks whose dW is written, then added, into one fp32 tensor: each
    chunk's own fp16 gradient widened, and their sum."""
    from reversability_amd.kernels import padded_head, tied_head_ce
    rows, d, vocab = 300, 128, 1001
    g = torch.Generator().manual_seed(13)
    x16 = torch.randn(rows, d, generator=g).half().to(cuda_device)
    head16 = padded_head((0.05 * torch.randn(vocab, d, generator=g)).to(cuda_device))
    labels = torch.randint(0, vocab, (rows,), generator=g).to(cuda_device)
    grad = torch.tensor([0.37], device=cuda_device)
    out = torch.full((vocab * d + 4,), float("nan"), device=cuda_device)
    dw = out[offset:offset + vocab * d].view(vocab, d)
    total = None
    for i, part in enumerate((slice(0, 170), slice(170, rows))):
        args = (x16[part], head16, vocab, labels[part], grad)
        *_, alone = tied_head_ce(*args, dw_out=torch.empty(out.shape, device=cuda_device)[
            offset:offset + vocab * d].view(vocab, d))
        *_, got = tied_head_ce(*args, dw_out=dw, accumulate=i > 0)
        total = alone if total is None else total + alone
        assert got is dw and torch.equal(alone, alone.half().float())
        assert torch.equal(dw, total)
    assert torch.isnan(out[:offset]).all() and torch.isnan(out[offset + vocab * d:]).all()
