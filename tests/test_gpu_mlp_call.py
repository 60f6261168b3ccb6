"""fp8_mlp, gate_up_silu_quant and quantize_weight through their one-call
bindings: the bits, shapes and errors of the registered ops one by one, over
the row counts where the gate/up GEMM changes how it gets its codes."""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from hf_kernels_helion_amd import finegrained_fp8_helion as fp8
from hf_kernels_helion_amd.finegrained_fp8_helion import synthetic

pytestmark = pytest.mark.gpu


class _Ops(TorchDispatchMode):
    """Active, it makes the calls take the registered ops one by one."""

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def _weights(H, I, dev):
    w13, s13 = [t.to(dev) for t in synthetic.weights(2 * I, H, seed=42)]
    w2, s2 = [t.to(dev) for t in synthetic.weights(H, I, seed=43)]
    return w13, s13, w2, s2


@pytest.mark.parametrize("M", [0, 1, 8, 17, 33, 64, 300, 511, 512, 700])
@pytest.mark.parametrize("interleaved,fuse", [(False, True), (False, False), (True, True)])
@pytest.mark.parametrize("H,I", [(1024, 1536), (4096, 512)])
def test_one_call_equals_ops(M, interleaved, fuse, H, I, dev):
    print(f"fp8_mlp one call M={M} H={H} I={I} {interleaved} {fuse}", flush=True)
    x = synthetic.activations(max(M, 1), H, seed=M, outlier_frac=0.01).to(dev)[:M]
    w13, s13, w2, s2 = _weights(H, I, dev)
    if interleaved:
        w13, s13 = fp8.interleave_gate_up(w13, s13)
    call = lambda v: fp8.fp8_mlp(v, w13, s13, w2, s2, fuse_quant=fuse,
                                 gate_up_interleaved=interleaved)
    y = call(x)
    with _Ops():
        ref = call(x)
    assert y.shape == ref.shape == (M, H) and torch.equal(y, ref)
    if M == 64:
        xt = x.t().contiguous().t().view(4, 16, H)      # strided, leading dimensions
        assert torch.equal(call(xt), y.view(4, 16, H))
    if interleaved and M:
        q, s = fp8.act_quant(x, 128)
        a = fp8.gate_up_silu_quant(q, s, w13, s13)
        with _Ops():
            b = fp8.gate_up_silu_quant(q, s, w13, s13)
        assert torch.equal(a[0].view(torch.uint8), b[0].view(torch.uint8))
        assert torch.equal(a[1], b[1])


def test_other_types_widths_and_errors(dev):
    """fp32 and fp16 activations, widths that are not whole groups and other
    blocks keep the ops' route; what raised still raises."""
    H, I = 200, 256
    for dt in (torch.float32, torch.float16, torch.bfloat16):
        x = synthetic.activations(5, H, seed=1).to(dt).to(dev)
        w13, s13, w2, s2 = _weights(H, I, dev)
        y = fp8.fp8_mlp(x, w13, s13, w2, s2)
        with _Ops():
            ref = fp8.fp8_mlp(x, w13, s13, w2, s2)
        assert torch.equal(y, ref)
    w13, s13, w2, s2 = _weights(512, I, dev)
    x = synthetic.activations(5, 512, seed=1).to(dev)
    with pytest.raises(RuntimeError):
        fp8.fp8_mlp(x[:, :256], w13, s13, w2, s2)
    with pytest.raises(RuntimeError):
        fp8.fp8_mlp(x.cpu(), w13, s13, w2, s2)
    with pytest.raises(RuntimeError):
        fp8.fp8_mlp(x, w13.float(), s13, w2, s2)
    with pytest.raises(RuntimeError, match="multiple of 128"):
        fp8.fp8_mlp(x, w13[:384], s13[:3], w2, s2, gate_up_interleaved=True)
    with pytest.raises(ValueError):
        fp8.fp8_mlp(x, w13, s13, w2, s2, block_size=(64, 128), gate_up_interleaved=True)
    W = torch.randn(300, 520, device=dev)
    a = fp8.quantize_weight(W)
    with _Ops():
        b = fp8.quantize_weight(W)
    assert torch.equal(a[0].view(torch.uint8), b[0].view(torch.uint8)) and torch.equal(a[1], b[1])
    with pytest.raises(RuntimeError):
        fp8.quantize_weight(W, (64, 64))
