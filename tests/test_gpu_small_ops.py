"""GPU parity of the small fused ops through the C ABI.  Bars: bf16 outputs
within 1 bf16 ulp of the oracle (the kernels may contract a*b+c into one
FMA), residual sums, KV copies, gathers, argmax and the step advance exact."""
import numpy as np
import pytest

from oracle import ops as oops
from oracle.bf16 import bf16_bits_to_f32, f32_to_bf16_bits

from _util import bf16_dev, bf16_ulp_diff, bits_of, f32_of, pkg, randn_bf16

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    import torch
    return torch.device("cuda:0")


@pytest.fixture(scope="module")
def ops():
    return pkg("native.torch_ops")


@pytest.mark.parametrize("rows,hidden", [(1, 2560), (3, 2560), (2, 4096), (1, 8), (1, 16384)])
@pytest.mark.parametrize("with_residual", [True, False])
def test_add_rmsnorm(ops, dev, rows, hidden, with_residual):
    rng = np.random.default_rng(rows * hidden)
    x = randn_bf16(rng, (rows, hidden))
    r = randn_bf16(rng, (rows, hidden), 3.0)
    g = f32_to_bf16_bits((1 + 0.1 * rng.standard_normal(hidden)).astype(np.float32))
    y, ro = ops.add_rmsnorm(bf16_dev(x, dev), bf16_dev(r, dev) if with_residual else None,
                            bf16_dev(g, dev), 1e-6)
    ry, rro = oops.add_rmsnorm(bf16_bits_to_f32(x), bf16_bits_to_f32(r) if with_residual else None,
                               bf16_bits_to_f32(g), 1e-6)
    assert bf16_ulp_diff(bits_of(y).reshape(rows, hidden), f32_to_bf16_bits(ry)).max() <= 1
    np.testing.assert_array_equal(bits_of(ro).reshape(rows, hidden), f32_to_bf16_bits(rro))


def test_add_rmsnorm_in_place_residual(ops, dev):
    rng = np.random.default_rng(1)
    x = randn_bf16(rng, (1, 2560))
    r = randn_bf16(rng, (1, 2560))
    g = randn_bf16(rng, 2560)
    rt = bf16_dev(r, dev)
    y, ro = ops.add_rmsnorm(bf16_dev(x, dev), rt, bf16_dev(g, dev), 1e-6, residual_out=rt)
    _, rro = oops.add_rmsnorm(bf16_bits_to_f32(x), bf16_bits_to_f32(r), bf16_bits_to_f32(g), 1e-6)
    np.testing.assert_array_equal(bits_of(rt).reshape(1, 2560), f32_to_bf16_bits(rro))


def test_qknorm_rope_kv_write(ops, dev):
    import torch
    rng = np.random.default_rng(3)
    n_q, n_kv, hd, bs, nblk, T = 32, 8, 128, 128, 6, 3
    nh = n_q + 2 * n_kv
    qkv = randn_bf16(rng, (T, nh * hd))
    qg = f32_to_bf16_bits((1 + 0.1 * rng.standard_normal(hd)).astype(np.float32))
    kg = f32_to_bf16_bits((1 + 0.1 * rng.standard_normal(hd)).astype(np.float32))
    cs = f32_to_bf16_bits(oops.rope_cache(8192, hd, 1e6))
    positions = np.array([0, 4095, 7000], dtype=np.int64)
    slots = np.array([5, 130, -1], dtype=np.int64)
    kc = torch.zeros((nblk, bs, n_kv, hd), dtype=torch.bfloat16, device=dev)
    vc = torch.zeros_like(kc)
    q_out = ops.qknorm_rope_kv_write(bf16_dev(qkv, dev), bf16_dev(qg, dev), bf16_dev(kg, dev),
                                     bf16_dev(cs, dev), torch.from_numpy(positions).to(dev),
                                     torch.from_numpy(slots).to(dev), kc, vc, n_q, n_kv, 1e-6)
    qkvf = bf16_bits_to_f32(qkv).reshape(T, nh, hd)
    csf = bf16_bits_to_f32(cs)
    kcb = bits_of(kc).reshape(nblk * bs, n_kv, hd)
    vcb = bits_of(vc).reshape(nblk * bs, n_kv, hd)
    qo = bits_of(q_out).reshape(T, n_q, hd)
    for t in range(T):
        row = csf[positions[t]]
        rq = oops.apply_rope(oops.rms_norm(qkvf[t, :n_q], bf16_bits_to_f32(qg), 1e-6), row)
        assert bf16_ulp_diff(qo[t], f32_to_bf16_bits(rq)).max() <= 1
        rk = oops.apply_rope(oops.rms_norm(qkvf[t, n_q:n_q + n_kv], bf16_bits_to_f32(kg), 1e-6), row)
        if slots[t] >= 0:
            assert bf16_ulp_diff(kcb[slots[t]], f32_to_bf16_bits(rk)).max() <= 1
            np.testing.assert_array_equal(vcb[slots[t]], qkv.reshape(T, nh, hd)[t, n_q + n_kv:])
    written = set(int(s) for s in slots if s >= 0)
    for s in range(nblk * bs):
        if s not in written:
            assert not kcb[s].any() and not vcb[s].any(), f"slot {s} written"


@pytest.mark.parametrize("rows,d", [(1, 9728), (4, 100)])
def test_silu_mul(ops, dev, rows, d):
    rng = np.random.default_rng(d)
    gu = randn_bf16(rng, (rows, 2 * d), 4.0)
    out = ops.silu_mul(bf16_dev(gu, dev))
    f = bf16_bits_to_f32(gu)
    ref = oops.silu_mul(f[:, :d], f[:, d:])
    assert bf16_ulp_diff(bits_of(out).reshape(rows, d), f32_to_bf16_bits(ref)).max() <= 1


def _off(t, shift):
    """t's values in a contiguous view that starts `shift` elements into its
    buffer: an odd shift rules 16-byte accesses out."""
    import torch
    buf = torch.empty(t.numel() + shift, dtype=t.dtype, device=t.device)
    buf[shift:] = t.reshape(-1)
    return buf[shift:].view(t.shape)


@pytest.mark.parametrize("rows,d", [(1, 8), (3, 40), (63, 2056), (2, 9728), (257, 8200),
                                    (33, 8200), (113, 8200), (114689, 8)])
@pytest.mark.parametrize("act", ["silu", "gelu"])
def test_gated_vector_kernel_equals_scalar(ops, dev, rows, d, act):
    """16-byte and element-wise kernels, bit for bit: sizes around a
    workgroup's chunks, one and four chunks a thread, and sizes that stay with
    the element-wise kernel (below 2^18 outputs for SiLU and 7 * 2^17 for GELU,
    whatever the alignment); nothing past the end."""
    import torch
    gu = torch.randn(rows, 2 * d, device=dev).mul_(4).to(torch.bfloat16)
    gu[0, 0], gu[-1, d - 1] = float("inf"), float("-inf")
    lut = ops.gelu_table(dev)
    f = (lambda x, o: ops.silu_mul(x, out=o)) if act == "silu" else (
        lambda x, o: ops.gelu_mul(x, lut, out=o))
    buf = torch.full((rows * d + 64,), -7.0, dtype=torch.bfloat16, device=dev)
    got = f(gu, buf[:rows * d])
    ref = f(_off(gu, 1), torch.empty(rows, d, dtype=torch.bfloat16, device=dev))
    np.testing.assert_array_equal(bits_of(got).reshape(-1), bits_of(ref).reshape(-1))
    assert bool((buf[rows * d:] == -7.0).all())


@pytest.mark.parametrize("T,n_q,n_kv", [(1, 4, 1), (5, 3, 1), (17, 32, 8), (3, 8, 2),
                                        (307, 3, 1), (308, 3, 1), (32, 32, 8), (129, 8, 2)])
def test_qknorm_vector_kernel_equals_scalar(ops, dev, T, n_q, n_kv):
    """The 16-lanes-a-head kernel against the wave-a-head one, bit for bit,
    with head counts that leave a partial wave and slots that are skipped, on
    both sides of the 1536 heads from which the first is taken."""
    import torch
    torch.manual_seed(T)
    nh = n_q + 2 * n_kv
    qkv = torch.randn(T, nh * 128, device=dev).to(torch.bfloat16)
    qg, kg = ((1 + 0.1 * torch.randn(128, device=dev)).to(torch.bfloat16) for _ in range(2))
    cs = torch.randn(64, 128, device=dev).to(torch.bfloat16)
    pos = torch.randint(-2, 70, (T,), device=dev)  # clamped to the table
    blocks = max(3, T // 32 + 2)
    slots = torch.randperm(32 * blocks, device=dev)[:T].clone()
    slots[T // 2] = -1 if T > 1 else slots[0]
    res = []
    for shift in (0, 1):
        kv = torch.zeros(2, blocks, 32, n_kv, 128, dtype=torch.bfloat16, device=dev)
        q = ops.qknorm_rope_kv_write(_off(qkv, shift), qg, kg, cs, pos, slots, kv[0], kv[1], n_q,
                                     n_kv, 1e-6)
        res.append((bits_of(q), bits_of(kv)))
    np.testing.assert_array_equal(res[0][0], res[1][0])
    np.testing.assert_array_equal(res[0][1], res[1][1])


@pytest.mark.parametrize("hidden", [8, 264, 2560, 2056, 4104])
def test_embedding_and_cache_vector_kernels(ops, dev, hidden):
    """Gathers and KV copies with 16-byte accesses equal torch's, and the
    element-wise kernels' (misaligned tensors)."""
    import torch
    table = torch.randn(37, hidden, device=dev).to(torch.bfloat16)
    ids = torch.tensor([36, 0, -1, 5, 37], device=dev)
    ref = table[ids.clamp(0, 36)] * ((ids >= 0) & (ids < 37)).to(torch.bfloat16)[:, None]
    slots = torch.tensor([9, -1, 0, 64, 31], device=dev)  # 64: past the cache
    key, val = (torch.randn(5, 2, hidden // 2, device=dev).to(torch.bfloat16) for _ in range(2))
    for shift in (0, 1):
        out = ops.embedding(_off(table, shift), ids)
        assert torch.equal(out.view(5, hidden), ref.abs() * ref.sign())
        kv = torch.zeros(2, 2, 32, 2, hidden // 2, dtype=torch.bfloat16, device=dev)
        ops.reshape_and_cache(_off(key, shift), _off(val, shift), kv[0], kv[1], slots)
        exp = torch.zeros_like(kv).view(2, 64, 2, hidden // 2)
        for t in (0, 2, 4):
            exp[0, slots[t]], exp[1, slots[t]] = key[t], val[t]
        assert torch.equal(kv.view_as(exp), exp)


def test_embedding(ops, dev):
    import torch
    rng = np.random.default_rng(7)
    table = randn_bf16(rng, (1000, 256))
    ids = np.array([0, 999, 17, -1, 1000], dtype=np.int64)
    out = bits_of(ops.embedding(bf16_dev(table, dev), torch.from_numpy(ids).to(dev))).reshape(5, 256)
    np.testing.assert_array_equal(out[:3], table[ids[:3]])
    assert not out[3:].any()


def test_argmax(ops, dev):
    import torch
    rng = np.random.default_rng(8)
    logits = randn_bf16(rng, (3, 151936))
    logits[1, 5] = logits[1, 77] = f32_to_bf16_bits(np.float32([100.0]))[0]  # tie -> lowest index
    logits[2, 1234] = 0x7FC0  # NaN wins
    out = ops.argmax(bf16_dev(logits, dev)).cpu().numpy()
    assert out[0] == np.argmax(bf16_bits_to_f32(logits[0]))
    assert out[1] == 5
    assert out[2] == 1234


@pytest.mark.parametrize("vocab", [1, 7, 8, 17, 8191, 65535, 65543])
@pytest.mark.parametrize("kind", ["randn", "zeros", "ties", "nan", "-inf"])
def test_argmax_edges(ops, dev, vocab, kind):
    """Rows that start 2 to 14 bytes past a 16-byte boundary, single elements
    around the chunks, zeros of both signs (equal), NaN of both signs (first
    one wins), the lowest value everywhere; in one launch and, from 65536
    elements on, in two."""
    import torch
    rng = np.random.default_rng(vocab)
    x = randn_bf16(rng, (8, vocab))
    if kind == "zeros":
        x &= 0x8000
    elif kind == "ties":
        x = f32_to_bf16_bits(rng.integers(-3, 3, (8, vocab)).astype(np.float32))
    elif kind == "nan":
        x[:, vocab // 2], x[:, vocab - 1] = 0xFFC0, 0x7FC0
    elif kind == "-inf":
        x[:] = 0xFF80
    f = bf16_bits_to_f32(x)
    want = [int(np.argmax(np.isnan(r))) if np.isnan(r).any() else int(np.argmax(r)) for r in f]
    xd = bf16_dev(x, dev)
    assert ops.argmax(xd).cpu().tolist() == want
    keys = torch.empty(ops.argmax_num_keys(8, vocab), dtype=torch.int64, device=dev)
    assert (keys.numel() > 0) == (vocab >= 65536)
    assert ops.argmax(xd, keys=keys).cpu().tolist() == want


@pytest.mark.parametrize("rows,vocab,keys,launch", [
    (32, 65536, True, "parts"), (33, 65536, True, "one"), (1, 65535, True, "one"),
    (1, 98304, False, "one"), (32, 98305, False, "parts"), (33, 98305, False, "one")])
def test_argmax_launches(ops, dev, monkeypatch, rows, vocab, keys, launch):
    import torch
    x = torch.randn(rows, vocab, device=dev).to(torch.bfloat16)
    k = (torch.empty(ops.argmax_num_keys(rows, vocab), dtype=torch.int64, device=dev) if keys
         else None)
    seen, real = [], ops.call
    monkeypatch.setattr(ops, "call", lambda name, *a: (seen.append(name), real(name, *a))[1])
    got = ops.argmax(x, keys=k)
    assert seen == [{"parts": "smx_argmax_bf16_parts", "one": "smx_argmax_bf16"}[launch]]
    xc = x.cpu().float()
    assert got.cpu().tolist() == [int((r == r.max()).nonzero()[0]) for r in xc]


def test_argmax_ragged_vocab(ops, dev):
    """vocab 1003: row 0 is 16-byte aligned (chunks of 8 values, then a
    3-element tail), the other rows are not (element by element)."""
    rng = np.random.default_rng(9)
    v = 1003
    logits = randn_bf16(rng, (5, v))
    big = f32_to_bf16_bits(np.float32([50.0]))[0]
    logits[0, 1001] = big                     # in the tail
    logits[1, 3] = logits[1, 1002] = big      # tie across rows' elements -> lowest index
    logits[2, 999] = logits[2, 1000] = big    # tie across the chunk / tail boundary
    logits[3, 0] = 0x7FC0                     # NaN first element
    out = ops.argmax(bf16_dev(logits, dev)).cpu().numpy()
    assert out.tolist()[:4] == [1001, 3, 999, 0]
    assert out[4] == np.argmax(bf16_bits_to_f32(logits[4]))


def test_decode_advance(ops, dev):
    import torch
    table = torch.tensor([[3, 9, 4], [7, 1, 2]], dtype=torch.int32, device=dev)
    ids = torch.tensor([1, 2], dtype=torch.int64, device=dev)
    nxt = torch.tensor([42, 43], dtype=torch.int64, device=dev)
    pos = torch.tensor([127, 5], dtype=torch.int64, device=dev)
    sl = torch.tensor([128, 6], dtype=torch.int32, device=dev)
    slots = torch.zeros(2, dtype=torch.int64, device=dev)
    toks = torch.full((2, 300), -1, dtype=torch.int64, device=dev)
    ops.decode_advance(nxt, ids, pos, sl, slots, table, 128, tokens_out=toks)
    assert ids.tolist() == [42, 43]
    assert pos.tolist() == [128, 6]
    assert sl.tolist() == [129, 7]
    assert slots.tolist() == [9 * 128 + 0, 7 * 128 + 6]
    assert toks[0, 128].item() == 42 and toks[1, 6].item() == 43
    # past the end of the block table the slot becomes -1
    pos.fill_(3 * 128 - 1)
    ops.decode_advance(nxt, ids, pos, sl, slots, table, 128)
    assert slots.tolist() == [-1, -1]


def test_decode_advance_gathers_next_embedding(ops, dev):
    """With an embedding table, the advance kernel leaves the embedding row of
    each row's new id (the argmax of its keys, or the forced token), zeros
    for an id outside the vocab; the ids and positions are as without it."""
    import torch
    rng = np.random.default_rng(3)
    vocab, hidden, rows = 50, 2560, 3
    table = randn_bf16(rng, (vocab, hidden))
    tdev = bf16_dev(table, dev).view(vocab, hidden)
    keys = torch.zeros((rows, 700), dtype=torch.int64, device=dev)
    # row r's best key sits at index 500 + r with id 7 * r; ids are encoded
    # as 0xffffffff - id in the low word under a positive value key
    for r in range(rows):
        keys[r, 500 + r] = (0x9000 << 32) | (0xFFFFFFFF - 7 * r)
    nxt = torch.zeros(rows, dtype=torch.int64, device=dev)
    ids = torch.zeros(rows, dtype=torch.int64, device=dev)
    pos = torch.tensor([3, 9, 0], dtype=torch.int64, device=dev)
    sl = pos.to(torch.int32) + 1
    slots = torch.zeros(rows, dtype=torch.int64, device=dev)
    table_bt = torch.arange(rows * 4, dtype=torch.int32, device=dev).view(rows, 4)
    forced = torch.full((rows, 16), -1, dtype=torch.int64, device=dev)
    forced[1, 10] = 49          # row 1 takes a forced token
    forced[2, 1] = vocab + 5    # row 2 a forced id outside the vocab
    flen = torch.tensor([0, 11, 2], dtype=torch.int32, device=dev)
    out = torch.full((rows, hidden), 7.0, dtype=torch.bfloat16, device=dev)
    ops.decode_advance(nxt, ids, pos, sl, slots, table_bt, 128, forced_ids=forced,
                       forced_len=flen, argmax_keys=keys.view(rows, -1), embed_table=tdev,
                       embed_out=out)
    assert nxt.tolist() == [0, 7, 14]
    assert ids.tolist() == [0, 49, vocab + 5]
    assert pos.tolist() == [4, 10, 1]
    got = bits_of(out).reshape(rows, hidden)
    np.testing.assert_array_equal(got[0], table[0])
    np.testing.assert_array_equal(got[1], table[49])
    assert np.all(got[2] == 0)
