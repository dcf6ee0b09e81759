"""The native host side (``lowbit_comm_amd._host``) in front of the public entry points: what it takes, what it leaves to the
validating path, and what it must not by-pass."""
import pytest
import torch

DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}


def values(n, dtype, seed, sigma=1e-3):
    return (torch.randn(n, generator=torch.Generator().manual_seed(seed)) * sigma).to(dtype)


# a lazily negated view is contiguous and has an address, but the memory there holds the negatives of its values
@pytest.mark.gpu
@pytest.mark.parametrize("n", [70, 128])
@pytest.mark.parametrize("wire, policy", [("portable", {}), ("native", {}), ("native", {"topk": 1})])
@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
def test_negated_views_quantize_as_the_values_they_stand_for(hip_device, dtype, wire, policy, n):
    from lowbit_comm_amd import CompressionConfig, quantize_tensor
    from lowbit_comm_amd.hip.loader import load_hip_extension
    from lowbit_comm_amd.quantization.codec import compensate_and_quantize

    status, config = load_hip_extension(wire_format=wire), CompressionConfig(**policy)
    x, r = (torch._neg_view(values(n, DTYPES[dtype], seed).to(hip_device)) for seed in (1, 2))
    assert x.is_neg() and x.is_contiguous()
    want = quantize_tensor(x.resolve_neg(), config, extension_status=status)
    assert torch.equal(quantize_tensor(x, config, extension_status=status), want)
    if n % 64 == 0:
        into = torch.zeros_like(want)
        assert torch.equal(quantize_tensor(x, config, extension_status=status, output=into), want)
    if not policy:
        into, sums = torch.zeros_like(want), quantize_tensor(x.resolve_neg() + r.resolve_neg(), config, extension_status=status)
        quantize_tensor(x, config, extension_status=status, output=into, residual=r)
        assert torch.equal(into, sums)
        assert compensate_and_quantize(x, x.resolve_neg(), config, extension_status=status) is None
        assert compensate_and_quantize(x.resolve_neg(), x, config, extension_status=status) is None


# the sum that the one launch writes has no history: operands that autograd follows keep torch's own add
@pytest.mark.gpu
def test_compensated_quantize_leaves_tangents_to_torch(hip_device):
    from lowbit_comm_amd import CompressionConfig
    from lowbit_comm_amd.hip.loader import load_hip_extension
    from lowbit_comm_amd.quantization.codec import compensate_and_quantize

    status, config = load_hip_extension(wire_format="native"), CompressionConfig()
    x, r, tangent = (values(128, torch.float32, seed).to(hip_device) for seed in (1, 2, 3))
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(x, tangent)
        assert compensate_and_quantize(dual, r, config, extension_status=status) is None
        assert compensate_and_quantize(r, dual, config, extension_status=status) is None
    assert compensate_and_quantize(x, r, config, extension_status=status) is not None


# no elements: the call succeeds without a device
def test_bound_launch_takes_a_stream_and_nothing_else():
    from lowbit_comm_amd.hip import ops

    nothing = (None, 0, None, -1, 0, 64, None, None, None, -1, None, 0, None, -1, 0)
    launch = ops.BoundLaunch("lbc_quant_pack", nothing, torch.device("cuda:0"), ())
    assert launch(0) is True and launch(stream=0) is True
    for args, kwargs in (((0, 0), {}), ((), {"streams": 0}), ((0,), {"stream": 0}), (("0",), {})):
        with pytest.raises(TypeError):
            launch(*args, **kwargs)


def modules():
    from lowbit_comm_amd.hip.cuda_wire_module import HipCudaWireModule
    from lowbit_comm_amd.hip.native_module import HipNativeModule

    return {"portable": HipNativeModule, "native": HipCudaWireModule}


# what the facade's allocating calls go through, method by method
CHAINS = [("portable", name, call) for call, names in {
    "quantize": ("quantize", "inplace_quantize", "inplace_quantize_pack"),
    "dequantize": ("dequantize", "inplace_dequantize"),
    "sum": ("dequantize_reduce", "inplace_dequantize_reduce"),
    "mean": ("dequantize_reduce_mean", "inplace_dequantize_reduce_mean")}.items() for name in names] + [
    ("native", name, call) for call, names in {
        "quantize": ("quantize", "inplace_quantize"), "compensate": ("quantize", "inplace_quantize"),
        "stochastic": ("philox_engine_inputs",), "dequantize": ("dequantize", "inplace_dequantize")}.items() for name in names]


@pytest.mark.gpu
@pytest.mark.parametrize("way", ["subclass", "class", "instance"])
@pytest.mark.parametrize("wire, name, call", CHAINS)
def test_a_replaced_method_is_asked(hip_device, monkeypatch, wire, name, call, way):
    from lowbit_comm_amd import CompressionConfig
    from lowbit_comm_amd.hip.loader import HipExtensionStatus, load_hip_extension
    from lowbit_comm_amd.quantization.codec import (compensate_and_quantize, dequantize_reduce_tensors, dequantize_tensor,
                                                    quantize_tensor)

    config = CompressionConfig(stochastic=call == "stochastic", allow_experimental=call == "stochastic")
    x = values(100 if wire == "portable" else 128, torch.float32, 1).to(hip_device)
    payload = quantize_tensor(x, CompressionConfig(), extension_status=load_hip_extension(wire_format=wire))
    cls, asked = modules()[wire], []
    before = cls.__dict__[name]
    own = before.__func__ if isinstance(before, staticmethod) else before

    def spy(*args, **kwargs):
        asked.append(args[1] if isinstance(args[0], cls) else args[0])
        return own(*args, **kwargs)

    spy_of_class = staticmethod(spy) if isinstance(before, staticmethod) else spy
    if way == "subclass":
        module = type("Sub", (cls,), {name: spy_of_class})()
    else:
        module = cls()
        if way == "class":
            monkeypatch.setattr(cls, name, spy_of_class)
        else:
            monkeypatch.setattr(module, name, spy if isinstance(before, staticmethod) else spy.__get__(module))
    status = HipExtensionStatus(available=True, module=module)
    if call in ("quantize", "stochastic"):
        quantize_tensor(x, config, extension_status=status)
    elif call == "compensate":
        assert compensate_and_quantize(x, x, config, extension_status=status) is None
        asked.append(None)
    elif call == "dequantize":
        dequantize_tensor(payload, tuple(x.shape), config, dtype="fp32", extension_status=status)
    else:
        dequantize_reduce_tensors([payload, payload], tuple(x.shape), config, dtype="fp32", extension_status=status, reduce=call)
    assert len(asked) == 1
    if call == "quantize":
        assert asked[0].numel() == 128          # whole groups, as every module but the one that pads by itself gets them


# the payloads of a reduce may be the rows of one tensor; another number of rows over the same bytes is another call
@pytest.mark.gpu
def test_rows_of_one_tensor_are_counted_on_every_call(hip_device):
    from lowbit_comm_amd import CompressionConfig, quantize_tensor

    module = modules()["portable"]()
    n, config = 256, CompressionConfig()
    rows = torch.stack([quantize_tensor(values(n, torch.float32, seed).to(hip_device), config) for seed in range(4)])
    policy = (64, 0, 8, module.QuantType.Linear)
    listed, out = torch.empty(64, device=hip_device), torch.empty(64, device=hip_device)
    for view in (rows.view(2, -1), rows, rows.view(2, -1), rows.view(8, -1)):
        module.inplace_dequantize_reduce(list(view), listed, *policy, False)
        module.inplace_dequantize_reduce(view, out, *policy, False)
        assert torch.equal(out, listed), tuple(view.shape)
    whole, feedback = torch.empty(n, device=hip_device), torch.empty(n, device=hip_device)
    for _ in range(2):
        assert module.inplace_dequantize_reduce_mean(rows, whole, *policy, False, 4)
        assert not module.inplace_dequantize_reduce_mean(rows.view(2, -1), whole, *policy, False, 4)
        fused = module.inplace_dequantize_reduce_mean_update_error_feedback
        assert fused(rows, whole, whole, feedback, *policy, False, 4)
        assert not fused(rows.view(2, -1), whole, whole, feedback, *policy, False, 4)


# the package may be imported first and built afterwards, in one process
def test_a_build_after_the_import_is_picked_up():
    import subprocess
    import sys
    from pathlib import Path

    script = """
import sys, torch
class NotBuilt:
    def find_spec(self, name, path=None, target=None):
        if name == "lowbit_comm_amd._host":
            raise ImportError("not built")
sys.meta_path.insert(0, NotBuilt())
import lowbit_comm_amd
from lowbit_comm_amd.exceptions import CCDLUnavailableError
from lowbit_comm_amd.hip import cuda_wire_module, library, native_module, ops
nothing = ("lbc_quant_pack", (None, 0, None, -1, 0, 64, None, None, None, -1, None, 0, None, -1, 0), torch.device("cuda:0"), ())
for make in (native_module.HipNativeModule, cuda_wire_module.HipCudaWireModule, lambda: ops.BoundLaunch(*nothing)):
    try:
        make()
        raise SystemExit("made without its native part")
    except CCDLUnavailableError as exc:
        assert "not built" in str(exc)
del sys.meta_path[0]
assert ops.BoundLaunch(*nothing)(0) is True
for module in (native_module.HipNativeModule(), cuda_wire_module.HipCudaWireModule()):
    try:
        module.quantize(torch.zeros(64), 64, 0, False, 8, module.QuantType.Linear, False)
        raise SystemExit("a CPU tensor was taken")
    except RuntimeError as exc:
        assert "GPU tensor" in str(exc), exc
"""
    done = subprocess.run([sys.executable, "-c", script], cwd=Path(__file__).resolve().parent.parent, capture_output=True, text=True,
                          timeout=100)
    assert done.returncode == 0, done.stderr


# the hook's one launch for bucket + residual stands for ErrorFeedbackState.compensate, which looks the residual up itself
@pytest.mark.parametrize("way", ["plain", "subclass", "class", "instance"])
@pytest.mark.parametrize("name", ["compensate", "get"])
def test_a_feedback_state_of_its_own_keeps_its_compensate_step(monkeypatch, name, way):
    from lowbit_comm_amd import CompressionConfig
    from lowbit_comm_amd.communication import ddp_hook
    from lowbit_comm_amd.communication.gather_reduce import GatheredPayloads
    from lowbit_comm_amd.hip.loader import HipExtensionStatus
    from lowbit_comm_amd.quantization.error_feedback import ErrorFeedbackState

    launched = []
    monkeypatch.setattr(ddp_hook, "compensate_and_quantize_in_one_launch", lambda *a, **k: launched.append(a))
    monkeypatch.setattr(ddp_hook, "quantize_tensor", lambda tensor, *a, **k: torch.zeros(68, dtype=torch.uint8))
    monkeypatch.setattr(ddp_hook, "dequantize_reduce_tensors", lambda *a, **k: torch.zeros(64))
    own = {"compensate": ErrorFeedbackState.compensate, "get": ErrorFeedbackState.get}[name]
    replacement = lambda self, *args: own(self, *args)  # noqa: E731
    feedback = (type("Own", (ErrorFeedbackState,), {name: replacement}) if way == "subclass" else ErrorFeedbackState)()
    if way == "instance":
        monkeypatch.setattr(feedback, name, replacement.__get__(feedback))
    elif way == "class":
        monkeypatch.setattr(ErrorFeedbackState, name, replacement)
    feedback.put(0, torch.ones(64))

    class Bucket:
        def index(self):
            return 0

        def buffer(self):
            return torch.ones(64)

    hook = ddp_hook.create_ddp_comm_hook(
        CompressionConfig(error_feedback=True), strategy="all_gather", error_feedback=feedback,
        extension_status=HipExtensionStatus(available=True, module=object()),
        native_inplace_dequantize_reduce_update_feedback=lambda *a, **k: False,
        all_gather=lambda local: GatheredPayloads([local.buffer], 1))
    hook(None, Bucket())
    assert len(launched) == (way == "plain")


# what a shape may be is torch's to say, also where the decode writes straight into it
@pytest.mark.gpu
@pytest.mark.parametrize("wire", ["portable", "native"])
@pytest.mark.parametrize("shape", [None, (True, 128), (1 << 62, 4), (1 << 33, 1 << 33), ..., (128.0,), (-1,)])
def test_shapes_that_torch_refuses_are_refused(hip_device, wire, shape):
    from lowbit_comm_amd import CompressionConfig
    from lowbit_comm_amd.hip.loader import load_hip_extension
    from lowbit_comm_amd.quantization.codec import dequantize_reduce_tensors, dequantize_tensor, quantize_tensor

    status, config = load_hip_extension(wire_format=wire), CompressionConfig()
    payload = quantize_tensor(values(128, torch.float32, 1).to(hip_device), config, extension_status=status)
    if shape == (-1,):       # torch's "as many as there are": accepted, with the last element trimmed away by the facade
        assert dequantize_tensor(payload, shape, config, dtype="fp32", extension_status=status).numel() == 127
        return
    for call in (lambda: dequantize_tensor(payload, shape, config, dtype="fp32", extension_status=status),
                 lambda: dequantize_reduce_tensors([payload] * 2, shape, config, dtype="fp32", extension_status=status, reduce="mean")):
        with pytest.raises((TypeError, RuntimeError)):
            call()
