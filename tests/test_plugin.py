"""The plugin entry point and the graph-safe custom ops (CPU: import
discipline, idempotence, fake-tensor shapes; GPU: the ops equal the direct
kernel calls bit for bit)."""
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

from _util import bits_of, pkg

ROOT = Path(__file__).resolve().parent.parent


def test_plugin_import_is_stdlib_only():
    code = (
        "import sys, importlib.util\n"
        f"sys.path.insert(0, {str(ROOT)!r})\n"
        "import __graft_entry__ as g\n"
        "spec = importlib.util.spec_from_file_location('p', g.PKG_DIR / 'plugin' / '__init__.py')\n"
        "m = importlib.util.module_from_spec(spec); spec.loader.exec_module(m)\n"
        "bad = [n for n in ('torch', 'numpy', 'vllm') if n in sys.modules]\n"
        "print(','.join(bad))\n")
    out = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, check=True)
    assert out.stdout.strip() == "", f"plugin import pulled in {out.stdout.strip()}"


@pytest.mark.parametrize("device,rows", [("cpu", 2), ("cpu", 16), ("meta", 3)])
def test_head_rows_off_the_gpu(device, rows):
    """Several rows where the kernels cannot run are a bf16 product with the
    tied weight; a weight of another type is refused as that product refuses it."""
    import torch
    head = pkg("integration.head")
    layer = torch.nn.Module()
    w = torch.randn(40, 64, dtype=torch.bfloat16, device=device)
    layer.weight = torch.nn.Parameter(w, requires_grad=False)
    layer.q4_0_head = torch.zeros(40, 36, dtype=torch.uint8, device=device)
    x = torch.randn(rows, 64, dtype=torch.bfloat16, device=device)
    y = head.Q4_0HeadMethod().apply(layer, x)
    assert tuple(y.shape) == (rows, 40) and y.device.type == device
    if device == "cpu":
        assert torch.equal(y, torch.nn.functional.linear(x, w))
        layer.weight = torch.nn.Parameter(w.float(), requires_grad=False)
        with pytest.raises(RuntimeError):
            head.Q4_0HeadMethod().apply(layer, x)


def test_torch_sees():
    """Which states keep a product a torch operation (CPU: it reads torch's
    state alone)."""
    import torch
    from torch.autograd import forward_ad
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode
    sees = pkg("integration.linear").torch_sees
    x, w = torch.ones(2, 3), torch.nn.Parameter(torch.ones(4, 3), requires_grad=False)

    class Function(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Sub(torch.Tensor):
        pass

    assert not sees(x) and not sees(x, w)
    g = x.clone().requires_grad_(True)
    assert sees(g) and sees(x, torch.nn.Parameter(w.data))
    with torch.no_grad():
        assert not sees(g)
    assert sees(x.as_subclass(Sub)) and sees(x, w.data.as_subclass(Sub))
    seen = []
    torch.func.vmap(lambda r: (seen.append(sees(r)), r)[1])(x)
    torch.func.grad(lambda r: (seen.append(sees(r)), r.sum())[1])(x)
    with forward_ad.dual_level():
        seen.append(sees(x))
    with Function():
        seen.append(sees(x))
    with Dispatch():
        seen.append(sees(x))
    torch.set_autocast_enabled("cuda", True)
    seen.append(sees(x))
    torch.set_autocast_enabled("cuda", False)
    with torch.device("cpu"), Function():
        seen.append(sees(x))
    assert seen == [True] * 7
    # a default device changes no product
    with torch.device("cpu"):
        assert not sees(x)
    old = torch.get_default_device()
    torch.set_default_device("cpu")
    try:
        assert not sees(x)
    finally:
        torch.set_default_device(None if old == torch.device("cpu") else old)
    assert not sees(x)


def test_register_is_idempotent():
    plugin = pkg("plugin")
    a = plugin.register()
    b = plugin.register()
    assert a is b
    assert a["ops"] == "smx"
    import torch
    assert hasattr(torch.ops.smx, "q4_0_gemv")


def test_fake_shapes():
    import torch
    from torch._subclasses.fake_tensor import FakeTensorMode
    pkg("plugin").register()
    with FakeTensorMode():
        x = torch.empty((1, 2560), dtype=torch.bfloat16)
        w = torch.empty((9728, 1440), dtype=torch.uint8)
        assert torch.ops.smx.q4_0_gemv(x, w, 9728, 2560).shape == (1, 9728)
        assert torch.ops.smx.q4_0_gemv_swiglu(x, w, 4864, 2560).shape == (1, 4864)
        lut = torch.empty(4096, dtype=torch.bfloat16)
        assert torch.ops.smx.q4_0_gemv_gelu(x, w, lut, 4864, 2560).shape == (1, 4864)
        y, r = torch.ops.smx.add_rmsnorm(x, x, torch.empty(2560, dtype=torch.bfloat16), 1e-6)
        assert y.shape == r.shape == (1, 2560)
        q = torch.empty((1, 32, 128), dtype=torch.bfloat16)
        kc = torch.empty((4, 128, 8, 128), dtype=torch.bfloat16)
        out = torch.ops.smx.splitkv_decode_attention(
            q, kc, kc, torch.empty((1, 4), dtype=torch.int32), torch.empty(1, dtype=torch.int32),
            4, 0.088)
        assert out.shape == (1, 32, 128)
        ids = torch.ops.smx.argmax(torch.empty((3, 1000), dtype=torch.bfloat16))
        assert ids.shape == (3,) and ids.dtype == torch.int64
        # the reference's per-layer seam: (y, residual) shaped like its inputs
        # (src/spark_vllm_ascend/integration/model.py:81-82)
        y, r = torch.ops.smx.layer_run(x, x, torch.empty(1, dtype=torch.int64),
                                       "model.layers.0.self_attn.attn")
        assert y.shape == r.shape == (1, 2560) and y.dtype == r.dtype == torch.bfloat16


@pytest.mark.gpu
def test_custom_ops_match_direct_calls():
    import torch
    pkg("plugin").register()
    ops = pkg("native.torch_ops")
    w_mod = pkg("integration.weights")
    dev = torch.device("cuda:0")
    w = w_mod.synthetic_q4_0(1024, 2560, 3, dev)
    x = torch.randn((1, 2560), device=dev).to(torch.bfloat16)
    np.testing.assert_array_equal(bits_of(torch.ops.smx.q4_0_gemv(x, w, 1024, 2560)),
                                  bits_of(ops.q4_0_gemv(x, w, 1024, 2560)))
    np.testing.assert_array_equal(bits_of(torch.ops.smx.q4_0_gemv_swiglu(x, w, 512, 2560)),
                                  bits_of(ops.q4_0_gemv_swiglu(x, w, 512, 2560)))
    lut = ops.gelu_table(dev)
    np.testing.assert_array_equal(bits_of(torch.ops.smx.q4_0_gemv_gelu(x, w, lut, 512, 2560)),
                                  bits_of(ops.q4_0_gemv_gelu(x, w, lut, 512, 2560)))
    logits = torch.randn((2, 5000), device=dev).to(torch.bfloat16).float().cpu()
    ids = torch.ops.smx.argmax(logits.to(torch.bfloat16).to(dev)).cpu()
    for r in range(2):  # the first index holding the row maximum
        top = logits[r].max()
        assert logits[r, ids[r]] == top and not (logits[r, :ids[r]] == top).any()
