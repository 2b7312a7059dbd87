"""GPU parity of smx_q4_0_gemm_rows (any row count, any K % 32 == 0): against
float64 products of the weights it multiplies (exact up to 16 rows, their bf16
roundings above), one-hot activations that must select weights bit for bit
(which pins the lane transposes, the two alignments of a block and the last
block of the matrix), every launch shape, and the linear that routes to it."""
import numpy as np
import pytest

from oracle import q4_0 as oq
from oracle.bf16 import bf16_bits_to_f32, f32_to_bf16_bits

from _util import bf16_dev, bits_of, f32_of, pkg, randn_bf16

pytestmark = pytest.mark.gpu

# (n, k) odd in each way: fewer columns than a tile, an odd number of blocks in
# the matrix (its last block read 2 bytes early), K of 1..3 blocks past a tile
SIZES = [(1, 32), (33, 96), (50, 160), (97, 32), (131, 2592), (256, 2560)]


@pytest.fixture(scope="module")
def dev():
    import torch
    return torch.device("cuda:0")


@pytest.fixture(scope="module")
def ops():
    return pkg("native.torch_ops")


def _w(blocks, dev):
    import torch
    return torch.from_numpy(np.ascontiguousarray(blocks).reshape(-1)).to(dev)


def _weights(blocks, n, k, rows):
    w = oq.dequant_f32(blocks, n, k).reshape(n, k)
    return w if rows <= 16 else bf16_bits_to_f32(f32_to_bf16_bits(w))


def _check(y, x, w):
    """fp32 sums of k products in any order (k 2^-24 of the absolute sum),
    rounded to bf16 (2^-8 covers the half ulp of 2^-9 either way)."""
    x64, w64 = bf16_bits_to_f32(x).astype(np.float64), w.astype(np.float64)
    ref = x64 @ w64.T
    bound = 2.0 ** -8 * np.abs(ref) + x.shape[1] * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64).T)
    bad = np.abs(y - ref) > bound
    assert not bad.any(), (np.argwhere(bad)[:4], y[bad][:4], ref[bad][:4])


@pytest.mark.parametrize("n,k", SIZES)
@pytest.mark.parametrize("m", [1, 5, 16, 17, 48, 65, 193, 257])
def test_rows_vs_float64(ops, dev, m, n, k):
    blocks = oq.make_blocks(n, k, seed=n + k + m)
    x = randn_bf16(np.random.default_rng(m + n + k), (m, k))
    y = f32_of(ops.q4_0_gemm_rows(bf16_dev(x, dev), _w(blocks, dev), n, k)).reshape(m, n)
    _check(y, x, _weights(blocks, n, k, m))


@pytest.mark.parametrize("n,k", SIZES)
@pytest.mark.parametrize("m", [16, 40])
def test_rows_one_hot_bits_and_bounds(ops, dev, m, n, k):
    import torch
    blocks = oq.make_blocks(n, k, seed=n, scale=1.0)
    cols = (np.arange(m) * 37 + k - m) % k
    x = np.zeros((m, k), dtype=np.uint16)
    x[np.arange(m), cols] = f32_to_bf16_bits(np.float32([1.0]))[0]
    y = torch.full((m * n + 64,), 7.0, dtype=torch.bfloat16, device=dev)
    ops.q4_0_gemm_rows(bf16_dev(x, dev), _w(blocks, dev), n, k, out=y[:m * n])
    want = f32_to_bf16_bits(oq.dequant_f32(blocks, n, k).reshape(n, k)[:, cols].T + np.float32(0))
    np.testing.assert_array_equal(bits_of(y)[:m * n].reshape(m, n) & 0x7FFF, want & 0x7FFF)
    np.testing.assert_array_equal(f32_of(y)[:m * n].reshape(m, n), bf16_bits_to_f32(want))
    assert (y[m * n:] == 7.0).all()


def test_rows_every_launch_shape():
    """Each launch shape, forced through its tuning switch (read once per
    process, so one child process runs them all)."""
    import subprocess
    import sys
    from pathlib import Path
    code = """
import os
os.environ.update(SMX_TUNE="1", SMX_ALLOW_UNVALIDATED="1")
import importlib
import torch
import __graft_entry__
ops = importlib.import_module(__graft_entry__.load_package().__name__ + ".native.torch_ops")
g = torch.Generator(device="cuda")
g.manual_seed(1)
for m, n, k in ((17, 130, 416), (150, 77, 1056)):
    w = torch.randint(0, 60, (n * k // 32 * 18,), generator=g, device="cuda", dtype=torch.uint8)
    x = torch.randn((m, k), generator=g, device="cuda").to(torch.bfloat16)
    wd, xd = ops.q4_0_dequant_bf16(w, n, k).cpu().double(), x.cpu().double()
    ref = xd @ wd.T
    bound = 2.0 ** -8 * ref.abs() + k * 2.0 ** -24 * (xd.abs() @ wd.abs().T)
    for shape in range(14):
        os.environ["SMX_ROWS_SHAPE"] = str(shape)
        print(m, n, k, shape, flush=True)
        y = ops.q4_0_gemm_rows(x, w, n, k).cpu().double()
        assert ((y - ref).abs() <= bound).all(), (m, n, k, shape)
print("ok")
"""
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=100,
                       cwd=Path(__file__).resolve().parent.parent)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout[-200:] + r.stderr[-800:]


def test_rows_infinities(ops, dev):
    """An infinite activation gives what a product with the weights gives."""
    n, k, m = 48, 256, 20
    blocks = oq.make_blocks(n, k, seed=3)
    x = randn_bf16(np.random.default_rng(4), (m, k))
    x[3, 100], x[7, 5] = 0x7F80, 0xFF80
    with np.errstate(invalid="ignore"):
        ref = bf16_bits_to_f32(x).astype(np.float64) @ _weights(blocks, n, k, m).astype(np.float64).T
    for rows in (m, 8):
        y = f32_of(ops.q4_0_gemm_rows(bf16_dev(x[:rows], dev), _w(blocks, dev), n, k))
        y = y.reshape(rows, n)
        np.testing.assert_array_equal(np.isnan(y), np.isnan(ref[:rows]))
        np.testing.assert_array_equal(np.isposinf(y), np.isposinf(ref[:rows]))


@pytest.mark.parametrize("m", [16, 40])
def test_rows_subnormal_scales_bits(ops, dev, m):
    """One-hot activations select weights of subnormal and extreme finite
    scales of both signs bit for bit (zeros by value)."""
    n, k = 48, 416
    blocks = oq.make_blocks(n, k, seed=21)
    scales = np.uint16([0x0001, 0x8001, 0x03FF, 0x83FF, 0x0400, 0x7BFF, 0xFBFF, 0x0000, 0x8000])
    view = blocks.reshape(n * k // 32, 18)
    view[:, :2] = scales[np.arange(len(view)) % len(scales)][:, None].view(np.uint8)
    cols = (np.arange(m) * 37 + 5) % k
    x = np.zeros((m, k), dtype=np.uint16)
    x[np.arange(m), cols] = 0x3F80
    y = ops.q4_0_gemm_rows(bf16_dev(x, dev), _w(blocks, dev), n, k)
    want = f32_to_bf16_bits(oq.dequant_f32(blocks, n, k).reshape(n, k)[:, cols].T + np.float32(0))
    np.testing.assert_array_equal(f32_of(y).reshape(m, n), bf16_bits_to_f32(want))


@pytest.mark.parametrize("m", [1, 16, 17, 40])
def test_rows_infinite_and_nan_scales(ops, dev, m):
    """Infinite and NaN scales: above 16 rows what a product with the
    dequantised weights gives, up to 16 what the GEMV gives a row (the scale
    times a block's sum); rows without one keep their bounds."""
    n, k = 50, 288
    blocks = oq.make_blocks(n, k, seed=22)
    view = blocks.reshape(n, k // 32, 18)
    for r, b, h in ((3, 0, 0x7C00), (7, 4, 0xFC00), (20, 8, 0x7E00), (49, 8, 0x7C00)):
        view[r, b, :2] = np.uint16([h]).view(np.uint8)
    special = np.isin(np.arange(n), (3, 7, 20, 49))
    x = randn_bf16(np.random.default_rng(m), (m, k))
    xd, wd = bf16_dev(x, dev).view(m, k), _w(blocks, dev)
    y = f32_of(ops.q4_0_gemm_rows(xd, wd, n, k)).reshape(m, n)
    if m <= 16:
        ref = np.stack([f32_of(ops.q4_0_gemv(xd[r], wd, n, k)).reshape(n) for r in range(m)])
    else:
        w = f32_of(ops.q4_0_dequant_bf16(wd, n, k)).reshape(n, k).astype(np.float64)
        with np.errstate(invalid="ignore"):
            ref = bf16_bits_to_f32(x).astype(np.float64) @ w.T
    assert not np.isfinite(ref[:, special]).any() and np.isfinite(ref[:, ~special]).all()
    np.testing.assert_array_equal(np.isnan(y), np.isnan(ref))
    np.testing.assert_array_equal(np.isposinf(y), np.isposinf(ref))
    np.testing.assert_array_equal(np.isneginf(y), np.isneginf(ref))
    with np.errstate(invalid="ignore"):
        w = _weights(blocks, n, k, m)
    _check(y[:, ~special], x, w[~special])


def test_linear_routes(dev):
    """Rows that autograd records keep the library product and its gradient,
    and rows of any alignment give the same result (which launch each state
    makes: test_linear_launches)."""
    import torch
    lin = pkg("integration.linear")
    n, k, m = 4001, 2592, 40
    layer = lin.Q4_0Linear(k, [n], device=dev)
    blocks = oq.make_blocks(n, k, seed=5)
    layer.qweight.data.copy_(_w(blocks, dev).view(n, -1))
    x = bf16_dev(randn_bf16(np.random.default_rng(6), (m, k)), dev).view(m, k)
    y = layer(x)
    xg = x.clone().requires_grad_(True)
    yg = layer(xg)
    assert yg.requires_grad
    yg.float().sum().backward()
    assert xg.grad is not None and not y.requires_grad
    torch.testing.assert_close(y.float(), yg.detach().float(), rtol=2.0 ** -6, atol=1e-2)
    off = torch.empty(m * k + 1, dtype=torch.bfloat16, device=dev)[1:].view(m, k).copy_(x)
    assert torch.equal(layer(off), y)  # 2-byte aligned rows
    assert torch.equal(layer(off[:5]), layer(x[:5]))


@pytest.mark.parametrize("m,n,k,fused", [
    (2, 300, 10016, True), (2, 300, 10272, False), (2, 1536, 10272, True),
    (3, 96, 40928, True), (3, 96, 41056, False), (4, 96, 41056, True)])
def test_linear_few_rows_launches(dev, monkeypatch, m, n, k, fused):
    """One launch or a GEMV per row where K % 64 != 0, on both sides of the line."""
    ops = pkg("native.torch_ops")
    layer = pkg("integration.linear").Q4_0Linear(k, [n], device=dev)
    blocks = oq.make_blocks(n, k, seed=n + m)
    layer.qweight.data.copy_(_w(blocks, dev).view(n, -1))
    x = randn_bf16(np.random.default_rng(m), (m, k))
    seen, real = [], ops.call
    monkeypatch.setattr(ops, "call", lambda name, *a: (seen.append(name), real(name, *a))[1])
    y = f32_of(layer(bf16_dev(x, dev).view(m, k))).reshape(m, n)
    assert seen == (["smx_q4_0_gemm_rows"] if fused else ["smx_q4_0_gemv"] * m)
    _check(y, x, _weights(blocks, n, k, m))


@pytest.mark.parametrize("state", ["plain", "no_grad", "default device", "autograd", "vmap",
                                   "forward mode", "autocast", "function mode"])
def test_linear_launches(dev, monkeypatch, state):
    """One launch for rows that torch only multiplies, a default device set or
    not; dequantisation and torch's product where torch has to see it."""
    import torch
    from torch.autograd import forward_ad
    from torch.overrides import TorchFunctionMode
    ops = pkg("native.torch_ops")
    n, k, m = 4001, 2592, 40
    layer = pkg("integration.linear").Q4_0Linear(k, [n], device=dev)
    layer.qweight.data.copy_(_w(oq.make_blocks(n, k, seed=5), dev).view(n, -1))
    x = bf16_dev(randn_bf16(np.random.default_rng(6), (m, k)), dev).view(m, k)
    want = layer(x).float()
    seen, real = [], ops.call
    monkeypatch.setattr(ops, "call", lambda name, *a: (seen.append(name), real(name, *a))[1])

    class Mode(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    if state == "plain":
        y = layer(x)
    elif state == "no_grad":
        with torch.no_grad():
            y = layer(x.clone().requires_grad_(True))
    elif state == "default device":
        with torch.device(dev):
            y = layer(x)
    elif state == "autograd":
        y = layer(x.clone().requires_grad_(True)).detach()
    elif state == "vmap":
        y = torch.func.vmap(layer)(torch.stack((x, x)))[1]
    elif state == "forward mode":
        with forward_ad.dual_level():
            d = forward_ad.unpack_dual(layer(forward_ad.make_dual(x, x)))
            assert torch.equal(d.primal, d.tangent)
            y = d.primal
    elif state == "autocast":
        with torch.autocast("cuda", dtype=torch.float16):
            y = layer(x)
        assert y.dtype == torch.float16
    else:
        with Mode():
            y = layer(x)
    fused = state in ("plain", "no_grad", "default device")
    assert seen == ["smx_q4_0_gemm_rows" if fused else "smx_q4_0_dequant_bf16"]
    torch.testing.assert_close(y.float(), want, rtol=2.0 ** -6, atol=1e-2)
    seen.clear()
    layer(x[:5])
    assert seen == ["smx_q4_0_gemm_rows"]


@pytest.mark.parametrize("rows,vocab,hidden,fused", [
    (8, 1000, 8192, True), (9, 1000, 8192, False), (12, 4000, 8192, True),
    (13, 4000, 8192, False), (12, 1000, 5120, True), (13, 1000, 5120, False),
    (16, 1000, 2560, True), (16, 65536, 4096, True), (17, 1000, 2560, False)])
def test_head_launches(dev, monkeypatch, rows, vocab, hidden, fused):
    """Which product each side of the line takes, both within their bounds."""
    import torch
    ops = pkg("native.torch_ops")
    g = torch.Generator(device=dev)
    g.manual_seed(rows)
    q = torch.randint(0, 60, (vocab, hidden // 32 * 18), generator=g, dtype=torch.uint8, device=dev)
    head = pkg("integration.head").TiedQ4_0Head(q, vocab, hidden)
    x = torch.randn((rows, hidden), generator=g, device=dev).to(torch.bfloat16)
    seen, real = [], ops.call
    monkeypatch.setattr(ops, "call", lambda name, *a: (seen.append(name), real(name, *a))[1])
    y = head.logits(x).float()
    assert seen == (["smx_q4_0_gemm"] if fused else [])
    xd, wd = x.double().cpu(), head.weight[:500].double().cpu()
    ref, mag = xd @ wd.T, xd.abs() @ wd.abs().T
    # weights exact or rounded to bf16 (2^-9 of each product), fp32 sums, bf16 out
    bound = 2.0 ** -8 * ref.abs() + (2.0 ** -9 + hidden * 2.0 ** -24) * mag
    assert ((y[:, :500].cpu().double() - ref).abs() <= bound).all()


@pytest.mark.parametrize("rows", [1, 2, 16])
def test_head_blocks_of_any_alignment(dev, rows):
    """Blocks 2 bytes past a 4-byte boundary, and blocks with a row stride (more
    than one row), which the batched kernel does not read."""
    import torch
    head_mod = pkg("integration.head")
    vocab, hidden = 1003, 320
    blocks = oq.make_blocks(vocab, hidden, seed=9)
    x = randn_bf16(np.random.default_rng(rows), (rows, hidden))
    xd = bf16_dev(x, dev).view(rows, hidden)
    head = head_mod.TiedQ4_0Head(_w(blocks, dev).view(vocab, -1), vocab, hidden)
    row = blocks.size // vocab
    wide = torch.zeros(vocab * row + 2, dtype=torch.uint8, device=dev)[2:].view(vocab, row)
    strided = torch.zeros(vocab, row + 4, dtype=torch.uint8, device=dev)[:, :row]
    for q in (wide, strided) if rows > 1 else (wide,):
        q.copy_(_w(blocks, dev).view(vocab, row))
        head.q4_0_head = q
        y = f32_of(head.logits(xd)).reshape(rows, vocab)
        _check(y, x, _weights(blocks, vocab, hidden, 1 if rows == 1 else 17))


@pytest.mark.parametrize("rows", [2, 7, 16, 17])
def test_head_rows(dev, rows):
    """2 to 16 rows of logits multiply the exact weights (any 2-D strides and
    alignment), more the tied bf16 ones, and rows autograd records keep their
    gradient."""
    import torch
    head_mod = pkg("integration.head")
    vocab, hidden = 1003, 320
    blocks = oq.make_blocks(vocab, hidden, seed=9)
    head = head_mod.TiedQ4_0Head(_w(blocks, dev).view(vocab, -1), vocab, hidden)
    x = randn_bf16(np.random.default_rng(rows), (rows, hidden))
    xd = bf16_dev(x, dev).view(rows, hidden)
    y = head.logits(xd)
    _check(f32_of(y).reshape(rows, vocab), x, _weights(blocks, vocab, hidden, rows))
    wide = torch.zeros((rows, 2 * hidden + 1), dtype=torch.bfloat16, device=dev)
    wide[:, 1:hidden + 1] = xd
    assert torch.equal(head.logits(wide[:, 1:hidden + 1]), y)
    xg = xd.clone().requires_grad_(True)
    head.logits(xg).float().sum().backward()
    assert xg.grad is not None
