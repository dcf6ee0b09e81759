"""GPU tests of the host layer over the HIP kernels: the native-module shim behind the codec facade, the
codec callables, the bucket processor and comm hook, the precollected-payload executor, the
reduce-scatter plan and the workspace pool with real device events.  Expected values come from the CPU
oracle on the same inputs; integer/byte results and fp32 results are compared bit for bit."""
import numpy as np
import pytest
import torch

from lowbit_comm_amd import CompressionConfig
from lowbit_comm_amd.communication import FusedPayloadPacker, GatheredPayloads, PackedPayload, make_fused_payload_all_gather
from lowbit_comm_amd.communication.ddp import DDPBucketProcessor
from lowbit_comm_amd.communication.ddp_hook import create_ddp_comm_hook
from lowbit_comm_amd.quantization import ErrorFeedbackState, Quantizer, codec
from oracle import codec_np, codec_torch

pytestmark = pytest.mark.gpu
CFG = CompressionConfig()


@pytest.fixture(scope="module")
def dev(hip_device):
    return hip_device


@pytest.fixture(scope="module")
def status(dev):
    from lowbit_comm_amd.hip.loader import load_hip_extension

    found = load_hip_extension()
    assert found.available, found.reason
    return found


def grad(n, dtype, seed, dev, sigma=1e-3):
    gen = torch.Generator().manual_seed(seed)
    return (torch.randn(n, generator=gen) * sigma).to(dtype).to(dev)


def same_bits(a, b):
    a, b = a.detach().cpu().contiguous(), b.detach().cpu().contiguous()
    assert a.dtype == b.dtype and a.shape == b.shape, (a.dtype, b.dtype, a.shape, b.shape)
    view = torch.int32 if a.dtype == torch.float32 else torch.int16
    return torch.equal(a.view(view), b.view(view))


def oracle_packed(x_cpu, g=64):
    return codec_torch.pack(*codec_torch.quantize(x_cpu, g))


class Bucket:
    def __init__(self, tensor, index=0):
        self._tensor, self._index = tensor, index

    def buffer(self):
        return self._tensor

    def index(self):
        return self._index


# --------------------------------------------------------------------------- #
# facade over the native module
# --------------------------------------------------------------------------- #
@pytest.mark.parametrize("dtype,name", [(torch.float32, "fp32"), (torch.bfloat16, "bf16"), (torch.float16, "fp16")])
@pytest.mark.parametrize("n", [64, 1000, 65_537])
def test_facade_quantize_dequantize_round_trip(status, dev, dtype, name, n):
    x = grad(n, dtype, 10 + n, dev).reshape(-1)
    buffer = codec.quantize_tensor(x, CFG, extension_status=status)
    assert buffer.dtype == torch.uint8 and torch.equal(buffer.cpu(), oracle_packed(x.cpu()))
    restored = codec.dequantize_tensor(buffer, (n,), CFG, dtype=name, extension_status=status)
    want = codec_torch.dequantize(*codec_torch.quantize(x.cpu()), n, 64, name)
    assert same_bits(restored, want)
    out = codec.allocate_quantized_buffer(x, CFG, dtype=name)
    meta = {}
    assert codec.quantize_tensor(x, CFG, extension_status=status, output=out, metadata=meta) is out
    assert meta["fused_quant_pack"] is True and meta["original_numel"] == n
    assert torch.equal(out, buffer)
    q = Quantizer(CFG, dtype=name, extension_status=status)
    assert torch.equal(q.quantize(x, q.allocate_q(x)), buffer)
    assert same_bits(q.dequantize(buffer, (n,)), want)


@pytest.mark.usefixtures("steady_allocator_counter")
def test_inplace_calls_do_not_allocate_or_touch_inputs(status, dev):
    n = 1 << 20
    x = grad(n, torch.float32, 1, dev)
    residual = grad(n, torch.float32, 2, dev, sigma=1e-5)
    keep_x, keep_r = x.clone(), residual.clone()
    out = codec.allocate_quantized_buffer(x, CFG, dtype="fp32")
    workspace = codec.allocate_dequantized_buffer(x, (n,), CFG)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    pointers = (out.data_ptr(), workspace.data_ptr())
    for _ in range(3):
        assert codec.inplace_quantize_pack(x, out, residual, CFG, extension_status=status)
        assert codec.inplace_dequantize_reduce_mean([out, out], workspace, CFG, extension_status=status, reduce="mean")
    torch.cuda.synchronize()
    assert torch.cuda.memory_allocated() == before
    assert (out.data_ptr(), workspace.data_ptr()) == pointers
    assert torch.equal(x, keep_x) and torch.equal(residual, keep_r)
    assert torch.equal(out.cpu(), oracle_packed(keep_x.cpu() + keep_r.cpu()))


@pytest.mark.parametrize("world", [2, 8, 11])
@pytest.mark.parametrize("reduce", ["sum", "mean"])
def test_facade_dequantize_reduce_matches_the_left_fold(status, dev, world, reduce):
    n = 40_000
    peers = [grad(n, torch.float32, 100 + r, dev) for r in range(world)]
    buffers = [codec.quantize_tensor(p, CFG, extension_status=status) for p in peers]
    payloads = [codec_torch.quantize(p.cpu()) for p in peers]
    want = codec_torch.reduce_payloads(payloads, n, 64, "fp32", reduce)
    got = codec.dequantize_reduce_tensors(buffers, (n,), CFG, dtype="fp32", extension_status=status, reduce=reduce)
    assert same_bits(got, want)
    workspace = codec.allocate_dequantized_buffer(peers[0], (n,), CFG)
    got = codec.dequantize_reduce_tensors(buffers, (n,), CFG, dtype="fp32", extension_status=status,
                                          output=workspace, reduce=reduce)
    assert same_bits(got, want) and got.data_ptr() == workspace.data_ptr()
    fused = codec.inplace_dequantize_reduce_mean(buffers, workspace, CFG, extension_status=status, reduce=reduce)
    assert fused is (world <= 8)


def test_facade_error_feedback_calls(status, dev):
    n, world = 30_016, 4
    peers = [grad(n, torch.float32, 200 + r, dev) for r in range(world)]
    buffers = [codec.quantize_tensor(p, CFG, extension_status=status) for p in peers]
    prepared = grad(n, torch.float32, 250, dev)
    restored = torch.empty(n, device=dev)
    residual = torch.empty(n, device=dev)
    assert codec.inplace_dequantize_reduce_mean_update_error_feedback(
        buffers, prepared, restored, residual, CFG, extension_status=status, reduce="mean")
    want = codec_torch.reduce_payloads([codec_torch.quantize(p.cpu()) for p in peers], n, 64, "fp32", "mean")
    assert same_bits(restored, want) and same_bits(residual, prepared.cpu() - want)
    residual2 = torch.zeros(n, device=dev)
    got = codec.dequantize_reduce_update_error_feedback(buffers, prepared, residual2, (n,), CFG, dtype="fp32",
                                                        extension_status=status, reduce="mean")
    assert same_bits(got, want) and same_bits(residual2, prepared.cpu() - want)
    residual3 = torch.zeros(n, device=dev)
    codec.update_error_feedback_residual(prepared, restored, residual3, extension_status=status)
    assert same_bits(residual3, prepared.cpu() - want)
    with pytest.raises(RuntimeError, match="divisor must be > 0"):
        status.module.inplace_dequantize_reduce_mean(buffers, restored, 64, 0, 8, status.module.QuantType.Linear, False, 0)
    with pytest.raises(RuntimeError, match="same number of elements"):
        codec.inplace_dequantize_reduce_mean_update_error_feedback(
            buffers, prepared, restored, residual[:-1], CFG, extension_status=status)


def test_native_module_remembers_launches_by_address_without_pinning_or_going_stale(status, dev):
    """From the second call with the same addresses on, an in-place entry point replays its bound launch.  The memo
    must follow the data (same launch, new contents), must not keep tensors alive, and must not serve a call whose
    tensors differ in anything the binding depends on."""
    import weakref

    module = status.module
    linear = module.QuantType.Linear
    n, world = 64 * 700, 4

    def unpack(packed):
        raw = packed.cpu()
        return raw[:n].view(torch.int8), raw[n:].view(torch.float32)

    x = grad(n, torch.float32, 31, dev)
    payload = torch.empty(n // 64 * 68, dtype=torch.uint8, device=dev)
    before = len(module._launches)
    for seed in (32, 33, 34):                                   # same addresses, new contents every time
        x.copy_(grad(n, torch.float32, seed, dev))
        assert module.inplace_quantize_pack(x, payload, None, 64, 0, False, 8, linear, False)
        assert torch.equal(payload.cpu(), oracle_packed(x.cpu()))
    assert len(module._launches) == before + 1
    peers = [codec.quantize_tensor(grad(n, torch.float32, 40 + r, dev), CFG, extension_status=status) for r in range(world)]
    out = torch.empty(n, device=dev)
    checked = []
    eligible = module._fused_eligible
    module._fused_eligible = lambda *args: checked.append(1) or eligible(*args)
    try:
        for _ in range(3):
            assert module.inplace_dequantize_reduce_mean(peers, out, 64, 0, 8, linear, False, world)
    finally:
        del module._fused_eligible
    assert len(checked) == 1, "the second and third call replay the remembered launch without looking at the tensors again"
    want = codec_torch.reduce_payloads([unpack(p) for p in peers], n, 64, "fp32", "mean")
    assert same_bits(out, want)
    assert module.inplace_dequantize_reduce_mean(peers[::-1], out, 64, 0, 8, linear, False, world)   # another order: another key
    want_reversed = codec_torch.reduce_payloads([unpack(p) for p in peers[::-1]], n, 64, "fp32", "mean")
    assert same_bits(out, want_reversed)
    assert module.inplace_dequantize_reduce_mean(peers, out, 64, 0, 8, linear, False, 1)             # another divisor
    assert same_bits(out, codec_torch.reduce_payloads([unpack(p) for p in peers], n, 64, "fp32", "sum"))
    # a tensor at a remembered address that is not what was bound: validated again, and refused
    with pytest.raises(RuntimeError):
        module.inplace_quantize_pack(x, payload.view(torch.int8), None, 64, 0, False, 8, linear, False)
    strided = torch.empty(2 * payload.numel(), dtype=torch.uint8, device=dev)[::2]
    with pytest.raises(RuntimeError):
        module.inplace_quantize_pack(x, strided, None, 64, 0, False, 8, linear, False)
    assert module.inplace_dequantize_reduce_mean([p[:-68] for p in peers], out, 64, 0, 8, linear, False, world) is False
    # nothing is kept alive
    fresh = grad(n, torch.float32, 50, dev)
    alive = weakref.ref(fresh)
    assert module.inplace_quantize_pack(fresh, payload, None, 64, 0, False, 8, linear, False)
    torch.cuda.synchronize()
    del fresh
    assert alive() is None
    assert len(module._launches) <= module.launch_memo_entries
    # a launch bound under one access mode is not replayed for a call made under another
    from lowbit_comm_amd.hip import ops

    count = len(module._launches)
    with ops.access_mode("cached"):
        assert module.inplace_quantize_pack(x, payload, None, 64, 0, False, 8, linear, False)
        assert len(module._launches) == count + 1
        assert module.inplace_quantize_pack(x, payload, None, 64, 0, False, 8, linear, False)
        assert len(module._launches) == count + 1
    assert torch.equal(payload.cpu(), oracle_packed(x.cpu()))


def test_unsupported_policies_decline_instead_of_failing(status, dev):
    x = grad(1024, torch.float32, 3, dev)
    out = torch.empty(1024 // 64 * 68, dtype=torch.uint8, device=dev)
    for cfg in (CompressionConfig(topk=1), CompressionConfig(stochastic=True), CompressionConfig(quant_type="normal"),
                CompressionConfig(bit=4, allow_experimental=True)):
        assert codec.inplace_quantize_pack(x, out, None, cfg, extension_status=status) is False
        if not cfg.stochastic:                      # decoding does not depend on how rounding was done
            assert codec.inplace_dequantize_reduce_mean([out], torch.empty_like(x), cfg, extension_status=status) is False
    with pytest.raises(RuntimeError, match="invalid quantized payload size"):
        codec.inplace_quantize_pack(x, out[:-1], None, CFG, extension_status=status)


# --------------------------------------------------------------------------- #
# codec callables + packer + hook
# --------------------------------------------------------------------------- #
def test_hip_codec_callables_produce_the_portable_payload_and_pack_without_a_copy(dev):
    from lowbit_comm_amd.hip.codec import dequantize_tensor_hip, quantize_tensor_hip

    x = grad(10_000, torch.bfloat16, 7, dev).reshape(100, 100)
    payload = quantize_tensor_hip(x, CFG)
    w_codes, w_scales = codec_torch.quantize(x.cpu())
    assert isinstance(payload, PackedPayload) and payload.shape == (100, 100) and payload.dtype == "bf16"
    assert payload.buffer.dtype == torch.int8 and torch.equal(payload.buffer.cpu(), w_codes)
    assert same_bits(payload.metadata["scales"], w_scales) and payload.metadata["original_numel"] == 10_000
    packer = FusedPayloadPacker.from_payload(payload)
    packed = packer.pack(payload)
    assert packed.data_ptr() == payload.packed.data_ptr() and torch.equal(packed.cpu(), codec_torch.pack(w_codes, w_scales))
    again = packer.unpack(packed, shape=payload.shape, dtype="bf16")
    restored = dequantize_tensor_hip(again, (100, 100), CFG, "bf16")
    assert same_bits(restored, codec_torch.dequantize(w_codes, w_scales, 10_000, 64, "bf16").reshape(100, 100))
    with pytest.raises(ValueError, match="linear"):
        quantize_tensor_hip(x, CompressionConfig(quant_type="normal"))
    with pytest.raises(ValueError, match="bit=8"):
        quantize_tensor_hip(x, CompressionConfig(bit=4, allow_experimental=True))


def _peer_gather(peers_cpu_payloads, dev):
    """all_gather stand-in: rank 0 is the local payload, the others are synthesised peers."""
    def all_gather(local):
        others = [CompressedPayloadOn(dev, codes, scales, local) for codes, scales in peers_cpu_payloads]
        return GatheredPayloads([local] + others, 1 + len(others))
    return all_gather


def CompressedPayloadOn(dev, codes, scales, like):
    from lowbit_comm_amd.communication import CompressedPayload

    return CompressedPayload(buffer=codes.to(dev), shape=like.shape, dtype=like.dtype,
                             metadata={"scales": scales.to(dev), "original_numel": like.metadata["original_numel"]})


@pytest.mark.parametrize("reduce", ["mean", "sum"])
def test_all_gather_hook_with_hip_callables_matches_the_reference_sequence(dev, reduce):
    from lowbit_comm_amd.hip.codec import dequantize_tensor_hip, quantize_tensor_hip

    n, world = 20_000, 4
    peers = [codec_torch.quantize(grad(n, torch.float32, 300 + r, "cpu")) for r in range(world - 1)]
    state = ErrorFeedbackState()
    hook = create_ddp_comm_hook(CFG, strategy="all_gather", reduce=reduce, quantize=quantize_tensor_hip,
                                dequantize=dequantize_tensor_hip, all_gather=_peer_gather(peers, dev),
                                error_feedback=state)
    cpu_residual = None
    for step in range(3):
        g = grad(n, torch.float32, 400 + step, dev)
        restored = hook(None, Bucket(g, index=5)).wait()
        prepared = g.cpu() if cpu_residual is None else g.cpu() + cpu_residual
        payloads = [codec_torch.quantize(prepared)] + peers
        want = codec_torch.reduce_payloads(payloads, n, 64, "fp32", reduce)
        cpu_residual = prepared - want
        assert same_bits(restored, want), f"step {step}"
        assert same_bits(state.get(5), cpu_residual), f"residual step {step}"


def test_all_gather_hook_facade_path_uses_the_fused_kernels(status, dev):
    """dequantize=None: flat uint8 buffers, fused decode+reduce, and from the second step on the fused
    decode+reduce+residual-update kernel into a cached workspace."""
    n, world = 50_000, 8
    peers = [oracle_packed(grad(n, torch.float32, 500 + r, "cpu")).to(dev) for r in range(world - 1)]
    peer_payloads = [codec_torch.quantize(grad(n, torch.float32, 500 + r, "cpu")) for r in range(world - 1)]

    def all_gather(local):
        return GatheredPayloads([local.buffer] + peers, world)

    state = ErrorFeedbackState()
    hook = create_ddp_comm_hook(CFG, strategy="all_gather", reduce="mean", all_gather=all_gather,
                                error_feedback=state, extension_status=status)
    cpu_residual = None
    outputs = []
    for step in range(4):
        g = grad(n, torch.float32, 600 + step, dev)
        restored = hook(None, Bucket(g, index=1)).wait()
        outputs.append(restored.data_ptr())
        prepared = g.cpu() if cpu_residual is None else g.cpu() + cpu_residual
        want = codec_torch.reduce_payloads([codec_torch.quantize(prepared)] + peer_payloads, n, 64, "fp32", "mean")
        cpu_residual = prepared - want
        assert same_bits(restored, want), f"step {step}"
        assert same_bits(state.get(1), cpu_residual), f"residual step {step}"
    assert outputs[1] == outputs[2] == outputs[3]          # cached decode workspace from step 1 on


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.usefixtures("steady_allocator_counter")
def test_all_gather_hook_takes_bucket_plus_residual_from_the_quantize_launch(status, dev, dtype):
    """With error feedback the reference's hook first forms ``prepared = bucket + residual`` in a kernel of its own
    (ccdl_comm/communication/ddp_hook.py:196; error_feedback.py:27-36) and needs it again after the gather.  Here
    the quantize launch writes it: same results as the hook with the compensate step left to torch (an injected
    quantizer switches the fusion off), two codec launches per bucket and no other kernel, nothing allocated from the
    third step on."""
    from torch.profiler import ProfilerActivity, profile

    n, world, buckets = 64 * 900, 4, 3
    peers = [[codec.quantize_tensor(grad(n, dtype, 800 + 10 * b + r, dev), CFG, extension_status=status)
              for r in range(world - 1)] for b in range(buckets)]
    current = [0]

    def all_gather(local):
        return GatheredPayloads([local.buffer] + peers[current[0]], world)

    states = [ErrorFeedbackState(), ErrorFeedbackState()]
    fused = create_ddp_comm_hook(CFG, strategy="all_gather", reduce="mean", all_gather=all_gather, error_feedback=states[0],
                                 extension_status=status, workspace_cache_max_entries=8)
    plain = create_ddp_comm_hook(CFG, strategy="all_gather", reduce="mean", all_gather=all_gather, error_feedback=states[1],
                                 extension_status=status, workspace_cache_max_entries=8,
                                 quantize=lambda tensor, active: codec.quantize_tensor(tensor, active, extension_status=status))
    grads = [grad(n, dtype, 850 + b, dev) for b in range(buckets)]
    allocated = None
    for step in range(5):
        for b in range(buckets):
            grads[b].copy_(grad(n, dtype, 900 + 10 * step + b, dev))
        torch.cuda.synchronize()
        if step == 3:
            allocated = torch.cuda.memory_allocated()
        with profile(activities=[ProfilerActivity.CUDA]) as prof:
            got = []
            for b in range(buckets):
                current[0] = b
                got.append(fused(None, Bucket(grads[b], index=b)).wait())
            torch.cuda.synchronize()
        kernels = [e.name for e in prof.events() if e.device_type == torch.autograd.DeviceType.CUDA
                   and "Memcpy" not in e.name and "Memset" not in e.name]
        if step >= 2:            # step 0 has no residual yet, step 1 creates the workspaces
            assert len(kernels) == 2 * buckets and all("lbc" in name for name in kernels), kernels
        if step == 4:
            assert torch.cuda.memory_allocated() == allocated
        for b in range(buckets):
            current[0] = b
            want = plain(None, Bucket(grads[b].clone(), index=b)).wait()
            assert got[b].dtype == want.dtype
            assert same_bits(got[b], want), f"bucket {b}, step {step}"
            assert same_bits(states[0].get(b), states[1].get(b)), f"residual {b}, step {step}"


def test_fused_all_gather_adapter_ships_one_packed_tensor(dev):
    from lowbit_comm_amd.hip.codec import dequantize_reduce_hip, quantize_tensor_hip

    n = 8192
    local = quantize_tensor_hip(grad(n, torch.float32, 1, dev), CFG)
    remote = quantize_tensor_hip(grad(n, torch.float32, 2, dev), CFG)
    seen = []

    def byte_all_gather(packed):
        seen.append((packed.data_ptr(), packed.numel()))
        return GatheredPayloads([packed, remote.packed], 2)

    gathered = make_fused_payload_all_gather(byte_all_gather)(local)
    assert seen == [(local.packed.data_ptr(), n // 64 * 68)]
    got = dequantize_reduce_hip(gathered.payloads, (n,), CFG, "fp32", "sum")
    want = codec_torch.reduce_payloads([(p.buffer.cpu(), p.metadata["scales"].cpu()) for p in (local, remote)], n)
    assert same_bits(got, want)
    assert dequantize_reduce_hip([local] * 9, (n,), CFG, "fp32", "sum") is None


# --------------------------------------------------------------------------- #
# fused local round trip (config 3 semantics)
# --------------------------------------------------------------------------- #
@pytest.mark.parametrize("dtype,name", [(torch.bfloat16, "bf16"), (torch.float32, "fp32"), (torch.float16, "fp16")])
def test_fused_bucket_processor_equals_the_unfused_reference_sequence(dev, dtype, name):
    n = 100_032
    fused = DDPBucketProcessor.from_hip_codec(CFG, fused=True)
    unfused = DDPBucketProcessor.from_hip_codec(CFG, fused=False)
    if dtype != torch.float32:                      # config 3: an fp32 residual already exists
        seed = grad(n, torch.float32, 9, dev, sigma=1e-5)
        fused.error_feedback.put(0, seed.clone())
        unfused.error_feedback.put(0, seed.clone())
        cpu_residual = seed.cpu()
    else:
        cpu_residual = None
    for step in range(4):
        g = grad(n, dtype, 700 + step, dev)
        torch.cuda.synchronize()
        out_fused = fused.process(Bucket(g), dtype=name)
        out_plain = unfused.process(Bucket(g), dtype=name)
        _c, _s, want, cpu_residual = codec_torch.ef_round_trip(g.cpu(), cpu_residual, 64, name)
        assert out_fused.dtype == dtype and same_bits(out_fused, want), f"step {step}"
        assert same_bits(out_plain, want), f"unfused step {step}"
        assert same_bits(fused.error_feedback.get(0), cpu_residual), f"residual step {step}"
        assert same_bits(unfused.error_feedback.get(0), cpu_residual), f"unfused residual step {step}"


@pytest.mark.usefixtures("steady_allocator_counter")
def test_fused_codec_steady_state_allocates_nothing(dev):
    from lowbit_comm_amd.hip.codec import FusedErrorFeedbackCodec

    n = 1 << 20
    fused = FusedErrorFeedbackCodec(CFG)
    g = grad(n, torch.bfloat16, 1, dev)
    fused.error_feedback.put("b", torch.zeros(n, device=dev))
    fused.step("b", g, "bf16")
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    residual_ptr = fused.error_feedback.get("b").data_ptr()
    for _ in range(5):
        payload, restored = fused.step("b", g, "bf16")
    torch.cuda.synchronize()
    assert torch.cuda.memory_allocated() == before
    assert fused.error_feedback.get("b").data_ptr() == residual_ptr
    assert payload.packed.numel() == n // 64 * 68 and restored.dtype == torch.bfloat16


# --------------------------------------------------------------------------- #
# precollected payloads (the reference's own "payloads already in device memory" entry)
# --------------------------------------------------------------------------- #
@pytest.mark.parametrize("world,fused", [(1, True), (8, True), (9, False)])
def test_precollected_payload_executor(status, dev, world, fused):
    from lowbit_comm_amd.hip.executors import FUSED_FAST_PATH, PrecollectedPayloadExecutor

    n = 64 * 500
    executor = PrecollectedPayloadExecutor(CFG, shape=(n,), dtype="fp32", extension_status=status)
    peers = [grad(n, torch.float32, 800 + r, "cpu") for r in range(world)]
    payloads = [oracle_packed(p).to(dev) for p in peers]
    prepared = grad(n, torch.float32, 850, dev)
    output = torch.empty(n, device=dev)
    residual = torch.empty(n, device=dev)
    assert executor.run_precollected_payloads(payloads, prepared, output, residual) is output
    want = codec_torch.reduce_payloads([codec_torch.quantize(p) for p in peers], n, 64, "fp32", "mean")
    assert same_bits(output, want) and same_bits(residual, prepared.cpu() - want)
    info = executor.last_execution_info
    assert info.fallback_used is (not fused)
    assert info.fast_path == (FUSED_FAST_PATH if fused else "python_fallback")
    if not fused:
        assert "at most 8 payloads" in info.fallback_reason
    assert executor.execution_counters.snapshot().completed_runs == 1
    with pytest.raises(ValueError, match="must contain"):
        executor.run_precollected_payloads([payloads[0][:-4]], prepared, output, residual)
    with pytest.raises(ValueError, match="must not be empty"):
        executor.run_precollected_payloads([], prepared, output, residual)
    assert executor.execution_counters.snapshot().failed_runs == 2


# --------------------------------------------------------------------------- #
# reduce-scatter plan with every rank simulated on one device (config 4 structure)
# --------------------------------------------------------------------------- #
@pytest.mark.parametrize("n,world", [(64 * 8 * 40, 8), (100_003, 4), (70_000, 3)])
def test_reduce_scatter_all_gather_plan_matches_the_oracle(dev, n, world):
    from lowbit_comm_amd.hip.reduce_scatter import ReduceScatterPlan, compressed_all_reduce_via_reduce_scatter

    buckets = [grad(n, torch.float32, 900 + r, dev) for r in range(world)]
    plans = [ReduceScatterPlan(n, torch.float32, world_size=world, rank=r, config=CFG, device=dev) for r in range(world)]
    for plan, bucket in zip(plans, buckets):
        plan.quantize_chunks(bucket)

    def all_to_all_for(rank):
        def exchange(received, send):
            for src in range(world):
                received[src].copy_(plans[src].send[rank])
        return exchange

    shards = []
    for r, plan in enumerate(plans):
        all_to_all_for(r)(plan.received, plan.send)
        reduced = plan.reduce_received(op="sum")
        assert reduced.metadata["fused_dequant_reduce"] and reduced.shard_index == r
        shards.append(reduced)
        plan.requantize_shard()

    def all_gather(gathered, mine):
        for src in range(world):
            gathered[src].copy_(plans[src].gathered[src])

    full = []
    for plan in plans:
        all_gather(plan.gathered, None)
        full.append(plan.decode_gathered())
    want_shards, want_full = codec_np.reduce_scatter_all_gather_plan([b.cpu().numpy() for b in buckets], 64, "sum")
    for r in range(world):
        assert np.array_equal(shards[r].shard.cpu().numpy().view(np.uint32), want_shards[r].view(np.uint32)), r
        assert np.array_equal(full[r].cpu().numpy().view(np.uint32), want_full.view(np.uint32)), r
    # the one-call form on rank 0, reusing its plan
    out = compressed_all_reduce_via_reduce_scatter(buckets[0], config=CFG, world_size=world, rank=0,
                                                   all_to_all=all_to_all_for(0), all_gather=all_gather, plan=plans[0])
    assert np.array_equal(out.cpu().numpy().view(np.uint32), want_full.view(np.uint32))


def test_asynchronous_shard_exchange_completes_through_the_pipeline(dev):
    """``compressed_reduce_scatter_shard(async_op=True)``: the exchange returns a work object, the shard is reduced
    when its future fires and arrives through a torch future, bit-identical to the synchronous call."""
    from lowbit_comm_amd.communication import AsyncShardPipeline
    from lowbit_comm_amd.hip.reduce_scatter import ReduceScatterPlan, compressed_reduce_scatter_shard

    world, n = 4, 64 * 4 * 300 + 11
    buckets = [grad(n, torch.float32, 950 + r, dev) for r in range(world)]
    plans = [ReduceScatterPlan(n, torch.float32, world_size=world, rank=r, config=CFG, device=dev) for r in range(world)]
    for plan, bucket in zip(plans[1:], buckets[1:]):
        plan.quantize_chunks(bucket)

    def copy_rows(received, send):
        received[0].copy_(send[0])
        for src in range(1, world):
            received[src].copy_(plans[src].send[0])

    class StartedExchange:
        """Stands in for the work of ``all_to_all_single(..., async_op=True)``: the copies are enqueued when the
        exchange starts; the future fires when the test lets it."""

        def __init__(self):
            self.future = torch.futures.Future()
            self.waited = 0

        def get_future(self):
            return self.future

        def wait(self):
            self.waited += 1

    started = []

    def start(received, send):
        copy_rows(received, send)
        started.append(StartedExchange())
        return started[-1]

    want = compressed_reduce_scatter_shard(buckets[0], config=CFG, world_size=world, rank=0, all_to_all=copy_rows)
    want_bits = want.shard.clone()
    advanced, fed = [], []
    work = compressed_reduce_scatter_shard(buckets[0], config=CFG, world_size=world, rank=0, all_to_all=start,
                                           plan=plans[0], async_op=True, update_feedback=fed.append,
                                           advance_policy=lambda: advanced.append(True))
    assert isinstance(work, AsyncShardPipeline) and work.query() is False and not fed
    assert buckets[0] in work.resources
    with pytest.raises(RuntimeError, match="has not been waited for"):   # one bucket in flight per plan
        plans[0].quantize_chunks(buckets[0])
    started[0].future.set_result(None)                          # the exchange is over
    assert work.query() is True and started[0].waited == 1 and advanced == [True]
    shard = work.wait()
    assert shard is fed[0] and shard.metadata["async_completion"] is True and shard.shard_index == 0
    torch.cuda.synchronize()
    assert same_bits(shard.shard, want_bits.cpu())
    with pytest.raises(TypeError, match="must return a work object"):
        compressed_reduce_scatter_shard(buckets[0], config=CFG, world_size=world, rank=0, all_to_all=copy_rows,
                                        plan=plans[0], async_op=True)


def test_reduce_scatter_plan_pins_no_caller_tensors_and_orders_uses_across_streams(hip_device):
    """A caller whose tensors are new every step must not have them pinned by the plan's cache of bound launches, a
    residual of another dtype at a recycled address must not reuse a stale binding, and a use of the plan on
    another stream is ordered after the previous use."""
    import weakref

    from lowbit_comm_amd.hip import ops
    from lowbit_comm_amd.hip.reduce_scatter import ReduceScatterPlan

    world, n = 4, 64 * 4 * 200
    config = CompressionConfig(error_feedback=False)
    plan = ReduceScatterPlan(n, torch.float32, world_size=world, rank=1, config=config, device=hip_device)
    kept = [torch.randn(n, device=hip_device) * 1e-3 for _ in range(6)]
    for bucket in kept:
        plan.quantize_chunks(bucket)
    assert len(plan._bound) == 6 <= ReduceScatterPlan._BOUND_LAUNCHES
    again = plan._bound[next(iter(plan._bound))]
    plan.quantize_chunks(kept[0])
    assert plan._bound[("q", kept[0].data_ptr(), None, None)] is again and len(plan._bound) == 6   # bound once per address
    fresh = torch.randn(n, device=hip_device)
    alive = weakref.ref(fresh)
    plan.quantize_chunks(fresh)
    torch.cuda.synchronize()
    del fresh
    assert alive() is None                                      # the cache did not keep the caller's tensor
    plan._BOUND_LAUNCHES = 4
    recycled, elsewhere = torch.randn(n, device=hip_device), torch.randn(n, device=hip_device)
    plan.quantize_chunks(recycled)                              # very likely the address `fresh` had: a hit
    plan.quantize_chunks(elsewhere)                             # a new address for sure
    assert len(plan._bound) == 4

    residual32 = torch.zeros(n, device=hip_device)
    residual16 = residual32.view(torch.bfloat16)[:n]            # same address, another dtype
    plan.quantize_chunks(kept[0], residual=residual32, new_residual=residual32)
    spec32 = (residual32.data_ptr(), torch.float32, n)
    assert ("q", kept[0].data_ptr(), spec32, spec32) in plan._bound
    with pytest.raises(RuntimeError):                           # no stale binding: bound anew, and refused (an fp32
        plan.quantize_chunks(kept[0], residual=residual16, new_residual=residual16)   # sum needs an fp32 residual out)

    want = plan.quantize_chunks(kept[3]).clone()
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        plan.quantize_chunks(kept[5])                           # the side stream now owns the plan's buffers
    assert plan._last_stream_handle == side.cuda_stream
    got = plan.quantize_chunks(kept[3])                         # back on the default stream: ordered after the side stream
    assert plan._last_stream_handle == ops.current_stream_handle(hip_device)
    torch.cuda.synchronize()
    assert torch.equal(got, want)


def test_reduce_scatter_plan_fused_requantize_matches_the_two_steps(hip_device):
    from lowbit_comm_amd.hip.reduce_scatter import ReduceScatterPlan, compressed_all_reduce_via_reduce_scatter

    world, n = 8, 8 * 64 * 500 + 1234
    config = CompressionConfig(error_feedback=False)
    buckets = [torch.randn(n, device=hip_device) * 1e-3 for _ in range(world)]
    plans = [ReduceScatterPlan(n, torch.float32, world_size=world, rank=r, config=config, device=hip_device)
             for r in range(world)]

    def all_to_all_for(rank):
        def exchange(received, send):
            for r in range(world):
                received[r].copy_(plans[r].send[rank])
        return exchange

    for r in range(world):
        plans[r].quantize_chunks(buckets[r])
    for mode in ("sum", "mean"):
        for r in (0, world - 1):
            all_to_all_for(r)(plans[r].received, plans[r].send)
            reduced = plans[r].reduce_received(op=mode)
            two_step = plans[r].requantize_shard(reduced.shard).clone()
            plans[r].gathered.zero_()
            fused = plans[r].reduce_and_requantize(op=mode)
            assert torch.equal(fused, two_step), (mode, r)

    def all_gather_for(rank):
        def gather(gathered, mine):
            for r in range(world):
                if r != rank:
                    all_to_all_for(r)(plans[r].received, plans[r].send)
                    gathered[r, :plans[r].payload_bytes].copy_(plans[r].reduce_and_requantize(op="mean"))
        return gather

    full_fused = compressed_all_reduce_via_reduce_scatter(buckets[0], config=config, world_size=world, rank=0,
                                                          all_to_all=all_to_all_for(0), all_gather=all_gather_for(0),
                                                          op="mean", plan=plans[0]).clone()
    full_kept = compressed_all_reduce_via_reduce_scatter(buckets[0], config=config, world_size=world, rank=0,
                                                         all_to_all=all_to_all_for(0), all_gather=all_gather_for(0),
                                                         op="mean", plan=plans[0], keep_shard=True)
    assert torch.equal(full_fused, full_kept)
    exact = torch.stack(buckets).mean(dim=0)
    assert float((full_fused - exact).norm() / exact.norm()) < 0.02


def test_asynchronous_plan_runs_on_the_communication_stream_and_completes_by_stream_wait(hip_device):
    """The whole plan enqueued behind a work object: same bits as the synchronous call; the launches land on the
    device's side stream (busy main stream: a long torch job is enqueued first and the work is handed back before
    it finished); ``wait()`` orders the current stream after the plan without blocking the host on it; the work
    keeps the plan and tensors referenced until released."""
    from lowbit_comm_amd.hip.completion import HipCompletionManager, communication_stream
    from lowbit_comm_amd.hip.reduce_scatter import (ReduceScatterPlan, compressed_all_reduce_async,
                                                    compressed_all_reduce_via_reduce_scatter)
    from lowbit_comm_amd.work import CompletionWork

    world, n = 4, 64 * 4 * 3000 + 77
    config = CompressionConfig(error_feedback=False)
    buckets = [torch.randn(n, device=hip_device) * 1e-3 for _ in range(world)]
    plans = [ReduceScatterPlan(n, torch.float32, world_size=world, rank=r, config=config, device=hip_device)
             for r in range(world)]
    for r in range(1, world):
        plans[r].quantize_chunks(buckets[r])

    def all_to_all(received, send):
        received[0].copy_(send[0])
        for r in range(1, world):
            received[r].copy_(plans[r].send[0])

    def all_gather(gathered, mine):
        for r in range(1, world):
            for src in range(world):
                plans[r].received[src].copy_(plans[0].send[r] if src == 0 else plans[src].send[r])
            gathered[r, :plans[r].payload_bytes].copy_(plans[r].reduce_and_requantize(op="mean"))

    want = compressed_all_reduce_via_reduce_scatter(buckets[0], config=config, world_size=world, rank=0,
                                                    all_to_all=all_to_all, all_gather=all_gather, op="mean",
                                                    plan=plans[0]).clone()
    torch.cuda.synchronize()
    manager = HipCompletionManager()
    big = torch.randn(4096, 4096, device=hip_device)
    for _ in range(20):
        big = big @ big * 1e-3                                   # keeps the main stream busy for a while
    out = torch.empty(n, device=hip_device)
    work = compressed_all_reduce_async(buckets[0], config=config, world_size=world, rank=0, all_to_all=all_to_all,
                                       all_gather=all_gather, op="mean", plan=plans[0], out=out, manager=manager)
    assert isinstance(work, CompletionWork)
    assert work.query() is False                                 # handed back while the device still works
    assert plans[0] in work.resources and buckets[0] is work.resources[0]
    side = communication_stream(torch.cuda)
    assert side != torch.cuda.current_stream(hip_device)
    result = work.wait()                                         # a device-side wait on the current stream
    doubled = result * 2                                         # ordered after the plan by that wait
    torch.cuda.synchronize()
    assert work.query() is True and result.data_ptr() == out.data_ptr()
    assert same_bits(result, want) and same_bits(doubled, want * 2)
    work.release_resources()
    assert work.resources == () and work.wait() is result


@pytest.mark.usefixtures("steady_allocator_counter")
def test_hook_over_the_reduce_scatter_transport_reuses_one_plan_per_bucket_shape(hip_device):
    """``create_ddp_comm_hook(strategy="reduce_scatter", reduce_scatter_all_gather=make_reduce_scatter_transport(...))``:
    every bucket runs the pre-bound plan, results equal the plan called directly, the bucket is reduced in place
    and steady-state steps allocate nothing."""
    from lowbit_comm_amd.hip.reduce_scatter import (ReduceScatterPlan, compressed_all_reduce_via_reduce_scatter,
                                                    make_reduce_scatter_transport)

    world = 4
    config = CompressionConfig(error_feedback=False)
    sizes = [64 * 4 * 700 + 5, 64 * 4 * 300]
    peers = {n: [ReduceScatterPlan(n, torch.float32, world_size=world, rank=r, config=config, device=hip_device)
                 for r in range(world)] for n in sizes}
    peer_data = {n: [torch.randn(n, device=hip_device) * 1e-3 for _ in range(world)] for n in sizes}
    for n in sizes:
        for r in range(1, world):
            peers[n][r].quantize_chunks(peer_data[n][r])

    def all_to_all(received, send):
        n = next(k for k in sizes if peers[k][0].row_stride == send.shape[1])
        received[0].copy_(send[0])
        for r in range(1, world):
            received[r].copy_(peers[n][r].send[0])

    def all_gather(gathered, mine):
        n = next(k for k in sizes if peers[k][0].row_stride == gathered.shape[1])
        for r in range(1, world):
            for src in range(world):
                peers[n][r].received[src].copy_(mine_send[n][r] if src == 0 else peers[n][src].send[r])
            gathered[r, :peers[n][r].payload_bytes].copy_(peers[n][r].reduce_and_requantize(op="mean"))

    mine_send = {}
    want = {}
    for n in sizes:                                     # the expected result, through the plan called directly
        probe = ReduceScatterPlan(n, torch.float32, world_size=world, rank=0, config=config, device=hip_device)
        mine_send[n] = probe.quantize_chunks(peer_data[n][0]).clone()
        want[n] = compressed_all_reduce_via_reduce_scatter(peer_data[n][0].clone(), config=config, world_size=world,
                                                           rank=0, all_to_all=all_to_all, all_gather=all_gather,
                                                           op="mean", plan=probe).clone()
    transport = make_reduce_scatter_transport(world_size=world, rank=0, all_to_all=all_to_all, all_gather=all_gather)
    hook = create_ddp_comm_hook(config, strategy="reduce_scatter", reduce="mean",
                                reduce_scatter_all_gather=transport)
    assert hook._ccdl_effective_strategy == "reduce_scatter"
    buckets = {n: Bucket(peer_data[n][0].clone(), i) for i, n in enumerate(sizes)}
    for n in sizes:
        result = hook(None, buckets[n]).wait()
        assert result.data_ptr() == buckets[n].buffer().data_ptr()          # reduced in place
        assert same_bits(result, want[n])
    assert len(transport.plans) == 2
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    for _ in range(3):
        for n in sizes:
            buckets[n].buffer().copy_(peer_data[n][0])
            assert same_bits(hook(None, buckets[n]).wait(), want[n])
    torch.cuda.synchronize()
    assert torch.cuda.memory_allocated() == before and len(transport.plans) == 2
    empty = hook(None, Bucket(torch.empty(0, device=hip_device), 9)).wait()         # an empty bucket is a no-op
    assert empty.numel() == 0
    with pytest.raises(ValueError, match="reduces in the bucket's dtype"):
        transport(buckets[sizes[0]].buffer(), config=config, op="mean", dtype="bf16")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_reduce_scatter_transport_with_local_error_feedback(hip_device, dtype):
    """Three steps of one bucket through the transport with error feedback: what is sent and the residual it keeps
    equal the oracle's compensate -> quantize -> residual cycle per destination chunk, step after step."""
    from lowbit_comm_amd.hip.reduce_scatter import make_reduce_scatter_transport

    world, g, n = 4, 64, 64 * 4 * 50 + 37
    config = CompressionConfig()
    sent = []

    def all_to_all(received, send):
        sent.append(send.clone())
        for r in range(world):
            received[r].copy_(send[0])

    def all_gather(gathered, mine):
        for r in range(world):
            gathered[r, :mine.numel()].copy_(mine)

    transport = make_reduce_scatter_transport(world_size=world, rank=0, all_to_all=all_to_all, all_gather=all_gather,
                                              error_feedback=True)
    bucket = torch.empty(n, dtype=dtype, device=hip_device)
    shard = -(-n // world)
    want_residual = torch.zeros(n)
    for step in range(3):
        x = grad(n, dtype, 40 + step, hip_device)
        bucket.copy_(x)
        result = transport(bucket, config=config, op="mean")
        assert result.data_ptr() == bucket.data_ptr()
        residual = next(iter(transport.residuals.values()))
        assert len(transport.residuals) == 1 and residual.dtype == torch.float32
        for d in range(world):
            piece = slice(d * shard, min(n, (d + 1) * shard))
            codes, scales, _restored, new_r = codec_torch.ef_round_trip(x[piece].cpu(), want_residual[piece], g, "fp32")
            row = sent[-1][d].cpu()
            padded = -(-shard // g) * g
            assert torch.equal(row[:codes.numel()].view(torch.int8), codes), (step, d)
            assert torch.equal(row[padded:padded + 4 * scales.numel()].view(torch.float32).view(torch.int32),
                               scales.view(torch.int32)), (step, d)
            want_residual[piece] = new_r
        assert same_bits(residual, want_residual), step
    transport.reset()
    assert not transport.residuals


def test_reduce_scatter_plan_beyond_eight_ranks_chains_exactly(dev):
    from lowbit_comm_amd.hip.reduce_scatter import ReduceScatterPlan

    n, world = 64 * 12 * 10, 12
    buckets = [grad(n, torch.float32, 950 + r, dev) for r in range(world)]
    plans = [ReduceScatterPlan(n, torch.float32, world_size=world, rank=r, config=CFG, device=dev) for r in range(world)]
    for plan, bucket in zip(plans, buckets):
        plan.quantize_chunks(bucket)
    for src in range(world):
        plans[0].received[src].copy_(plans[src].send[0])
    reduced = plans[0].reduce_received(op="mean")
    assert reduced.metadata["fused_dequant_reduce"] is False and "at most 8" in reduced.metadata["fused_dequant_reduce_reason"]
    shard = n // world
    payloads = [codec_np.quantize_chunks(b.cpu().numpy(), world, 64)[0] for b in buckets]
    want = codec_np.reduce_payloads(payloads, shard, 64, "fp32", "mean")
    assert np.array_equal(reduced.shard.cpu().numpy().view(np.uint32), want.view(np.uint32))


# --------------------------------------------------------------------------- #
# workspace pool with real streams and events
# --------------------------------------------------------------------------- #
@pytest.mark.usefixtures("steady_allocator_counter")
def test_pool_reuses_buffers_across_streams_without_host_sync(dev):
    from lowbit_comm_amd.hip import EventCompletion, WorkspaceKey, create_torch_workspace_pool

    pool = create_torch_workspace_pool()
    key = WorkspaceKey(backend="hip", collective="reduce_scatter", strategy="compressed", shape_class=(1 << 22,),
                       dtype="float32", world_size=8, bit=8, group_size=64, chunk_config=(0,), workspace_kind="reduced",
                       device=str(dev))
    producer, consumer = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(producer):
        lease = pool.acquire(key, producer)
        lease.buffer.fill_(1.0)
        for _ in range(20):
            lease.buffer.mul_(1.0000001)
        lease.release(completion=EventCompletion(producer))
    with torch.cuda.stream(consumer):
        taken = pool.acquire(key, consumer)            # same buffer: handed off (or idle if the work already ended)
        assert taken.buffer.data_ptr() == lease.buffer.data_ptr()
        total = taken.buffer.sum()
        taken.release(completion=EventCompletion(consumer))
    torch.cuda.synchronize()
    assert abs(float(total) / (1 << 22) - 1.0) < 1e-3
    stats = pool.stats
    assert (stats.hits, stats.misses) == (1, 1) and stats.in_flight_bytes == 0 and stats.cached_bytes == 4 << 22
    before = torch.cuda.memory_allocated()
    for _ in range(10):
        again = pool.acquire(key, torch.cuda.current_stream())
        again.release(completion=EventCompletion())
        torch.cuda.synchronize()
    assert torch.cuda.memory_allocated() == before and pool.stats.misses == 1


def test_bucket_stream_captured_in_a_hip_graph_replays_like_eager(dev):
    """The per-bucket launches allocate nothing and clear nothing, so a pass over many buckets can be captured in
    a HIP graph.  Four replays, with eager work and a synchronisation between them, must leave the same residuals,
    payload bytes and reduced shard as four eager passes from the same state (the residual update is in place, so
    every pass differs from the one before)."""
    from lowbit_comm_amd.hip import ops

    world, g, buckets, n = 8, 64, 6, 64 * 4096 + 64 * 8 * 5          # not a multiple of the block size
    shard = n // world
    stride = -(-ops.payload_nbytes(shard, g) // 256) * 256
    grads = grad(buckets * n, torch.bfloat16, 1, dev)
    start = grad(buckets * n, torch.float32, 2, dev, sigma=1e-5)
    residuals = start.clone()
    rows = torch.empty(world, stride, dtype=torch.uint8, device=dev)
    peers = [ops.quant_pack(grad(shard, torch.float32, 10 + r, dev), group_size=g) for r in range(world)]
    out = torch.empty(shard, device=dev)
    launches = []
    for i in range(buckets):
        piece = slice(i * n, (i + 1) * n)
        launches.append(ops.bind_quant_pack_chunks(grads[piece], rows, world, residual=residuals[piece],
                                                   new_residual=residuals[piece]))
        launches.append(ops.bind_dequant_reduce(peers, out, numel=shard))

    def one_pass():
        for launch in launches:
            assert launch()

    eager = []
    for _ in range(4):
        one_pass()
        torch.cuda.synchronize()
        eager.append((residuals.clone(), rows.clone(), out.clone()))
    residuals.copy_(start)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
        one_pass()
    torch.cuda.synchronize()
    residuals.copy_(start)                                            # capture enqueued nothing
    for want_residuals, want_rows, want_out in eager:
        graph.replay()
        torch.cuda.synchronize()
        assert same_bits(residuals, want_residuals) and torch.equal(rows, want_rows) and same_bits(out, want_out)
        assert float((torch.randn(1 << 16, device=dev) * 2).sum().item()) == pytest.approx(0.0, abs=1e4)   # eager work


def test_two_lane_bucket_stream_captured_in_a_hip_graph_replays_like_eager(dev):
    """The one-launch bucket steps dealt to two streams (fork, alternate, join) captured as one graph with two
    parallel branches: four replays with eager work between them against four eager one-stream passes."""
    from lowbit_comm_amd.hip import StreamLanes, ops

    world, g, buckets, n = 8, 64, 7, 64 * 8 * 520
    shard = n // world
    stride = -(-ops.payload_nbytes(shard, g) // 256) * 256
    grads = grad(buckets * n, torch.bfloat16, 21, dev)
    start = grad(buckets * n, torch.float32, 22, dev, sigma=1e-5)
    residuals = start.clone()
    rows = [torch.empty(world, stride, dtype=torch.uint8, device=dev) for _ in range(2)]       # one pair per lane
    outs = [torch.empty(shard, device=dev) for _ in range(2)]
    peers = [[ops.quant_pack(grad(shard, torch.float32, 30 + 8 * i + r, dev), group_size=g) for r in range(world)]
             for i in range(buckets)]
    launches, previous = [], None
    for i in range(buckets):
        piece = slice(i * n, (i + 1) * n)
        quant = ops.bind_quant_pack_chunks(grads[piece], rows[i & 1], world, residual=residuals[piece],
                                           new_residual=residuals[piece])
        reduce = ops.bind_dequant_reduce(peers[i], outs[i & 1], numel=shard)
        launches.append(quant if previous is None else ops.bind_quant_chunks_and_reduce(quant, previous))
        previous = reduce
    lanes = StreamLanes(2)

    def one_stream():
        for launch in launches:
            assert launch()
        assert previous()

    def two_lanes():
        lanes.fork()
        for i, launch in enumerate(launches):
            assert launch(lanes.handle(i))
        assert previous(lanes.handle(buckets))
        lanes.join()

    eager = []
    for _ in range(4):
        one_stream()
        torch.cuda.synchronize()
        eager.append((residuals.clone(), rows[0].clone(), rows[1].clone(), outs[0].clone(), outs[1].clone()))
    residuals.copy_(start)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
        two_lanes()
    torch.cuda.synchronize()
    residuals.copy_(start)                                            # capture enqueued nothing
    for want in eager:
        graph.replay()
        torch.cuda.synchronize()
        got = (residuals, rows[0], rows[1], outs[0], outs[1])
        assert all(torch.equal(a.view(torch.uint8), b.view(torch.uint8)) for a, b in zip(got, want))
        assert float((torch.randn(1 << 16, device=dev) * 2).sum().item()) == pytest.approx(0.0, abs=1e4)   # eager work


def test_stream_ordered_completion_records_nothing_while_a_buffer_stays_on_one_stream(dev):
    from lowbit_comm_amd.hip import StreamOrderedCompletion, WorkspaceKey, create_torch_workspace_pool

    pool = create_torch_workspace_pool()
    key = WorkspaceKey(backend="hip", collective="reduce_scatter", strategy="compressed", shape_class=(1 << 20,),
                       dtype="float32", world_size=8, bit=8, group_size=64, chunk_config=(0,), workspace_kind="reduced",
                       device=str(dev))
    main, other = torch.cuda.current_stream(), torch.cuda.Stream()
    completions = []
    first = None
    for step in range(5):                              # the same stream again and again: one buffer, no event, no wait
        lease = pool.acquire(key, main)
        first = first if first is not None else lease.buffer.data_ptr()
        assert lease.buffer.data_ptr() == first
        lease.buffer.fill_(float(step))
        completions.append(StreamOrderedCompletion(main))
        lease.release(completion=completions[-1])
    assert all(c._event is None for c in completions)
    assert pool.stats.misses == 1 and pool.stats.hits == 4
    assert completions[-1].covers(main) and not completions[-1].covers(other) and not completions[-1].peek()
    # another stream takes the buffer over: now the event exists, and the consumer is ordered after the fill
    with torch.cuda.stream(other):
        taken = pool.acquire(key, other)
        assert taken.buffer.data_ptr() == first
        total = taken.buffer.sum()
        taken.release(completion=StreamOrderedCompletion(other))
    assert completions[-1]._event is not None
    torch.cuda.synchronize()
    assert float(total) == 4.0 * (1 << 20)
    # query() answers for the host: it records (once) and becomes true when the stream has drained
    done = StreamOrderedCompletion(main)
    assert done.peek() is False
    done.synchronize()
    assert done.query() is True and done.peek() is True


@pytest.mark.usefixtures("steady_allocator_counter")
def test_llama_shaped_bucket_stream_through_the_pool(dev):
    """Config 5 structure at 1/64 scale: bf16 parameter tensors of a Llama-3-8B-shaped layer stack, flattened in
    reverse registration order into fixed-size buckets with a ragged tail; per bucket EF quant-pack and a W=8
    shard reduce with pooled workspaces.  Checks: bit parity of sampled buckets and of the ragged tail, pool
    misses == distinct workspace keys, zero allocations after the first pass."""
    from lowbit_comm_amd.hip import EventCompletion, ShardWorkspaceProvider, create_torch_workspace_pool
    from lowbit_comm_amd.hip import ops
    from lowbit_comm_amd.hip.codec import FusedErrorFeedbackCodec

    hidden, ffn, kv, vocab, layers = 512, 1792, 128, 16_032, 2
    shapes = [(vocab, hidden)]
    for _ in range(layers):
        shapes += [(hidden, hidden), (kv, hidden), (kv, hidden), (hidden, hidden), (ffn, hidden), (ffn, hidden),
                   (hidden, ffn), (hidden,), (hidden,)]
    shapes += [(hidden,), (vocab, hidden), (1001,)]      # the odd-sized last tensor makes the tail ragged
    total = sum(int(np.prod(s)) for s in shapes)
    bucket_numel = 1 << 20
    stream = torch.cat([grad(int(np.prod(s)), torch.bfloat16, 1000 + i, dev) for i, s in enumerate(reversed(shapes))])
    assert stream.numel() == total
    bounds = [(a, min(a + bucket_numel, total)) for a in range(0, total, bucket_numel)]
    assert (bounds[-1][1] - bounds[-1][0]) % 64 != 0          # ragged tail
    world = 8
    pool = create_torch_workspace_pool()
    provider = ShardWorkspaceProvider(pool, backend="hip", collective="reduce_scatter", strategy="compressed",
                                      device=str(dev))
    codec_ef = FusedErrorFeedbackCodec(CFG)
    cpu_residuals = {}

    def one_pass(check):
        for index, (a, b) in enumerate(bounds):
            bucket = stream[a:b]
            payload, _restored = codec_ef.step(index, bucket, "bf16")
            shard = -(-(b - a) // world)
            session = provider.begin(stream=torch.cuda.current_stream())
            received = [session.get_received_tensor_payload(index, r, bucket[:shard], CFG, dtype="bf16", world_size=world)
                        for r in range(world)]
            out = session.get_reduced_shard(index, torch.empty(0, dtype=torch.float32, device=dev), (shard,), CFG,
                                            dtype="fp32", world_size=world, rank=0)
            first = bucket[:shard].float()
            for r, row in enumerate(received):               # synthetic peers: scaled copies of this rank's chunk
                assert ops.quant_pack_payload_into(first * (1.0 + 0.125 * r), row)
            pairs = [ops.split_payload(row, shard) for row in received]
            assert ops.dequant_reduce_into(pairs, out, numel=shard)
            if check and index in (0, len(bounds) // 2, len(bounds) - 1):
                w_codes, w_scales, _r, cpu_residuals[index] = codec_torch.ef_round_trip(
                    bucket.cpu(), cpu_residuals.get(index), 64, "bf16")
                assert torch.equal(payload.buffer.cpu(), w_codes), index
                assert same_bits(payload.metadata["scales"], w_scales), index
                assert same_bits(codec_ef.error_feedback.get(index), cpu_residuals[index]), index
                peers = [codec_torch.quantize(first.cpu() * (1.0 + 0.125 * r)) for r in range(world)]
                assert same_bits(out[:shard], codec_torch.reduce_payloads(peers, shard)), index
            session.release(completion=EventCompletion())

    one_pass(check=True)
    torch.cuda.synchronize()
    distinct_keys = 2 * (world + 1)                           # full-size and tail shapes: W recv rows + 1 reduced each
    assert pool.stats.misses == distinct_keys
    before = torch.cuda.memory_allocated()
    one_pass(check=False)
    torch.cuda.synchronize()
    assert pool.stats.misses == distinct_keys
    assert torch.cuda.memory_allocated() <= before


# --------------------------------------------------------------------------- #
# HIP graph capture: the launches allocate nothing and never synchronise, so a bucket step can be captured
# --------------------------------------------------------------------------- #
def test_bucket_step_replays_from_a_hip_graph(dev):
    from lowbit_comm_amd.hip import ops
    from lowbit_comm_amd.hip.reduce_scatter import ReduceScatterPlan

    n, world = 64 * 8 * 500, 8
    plan = ReduceScatterPlan(n, torch.float32, world_size=world, rank=0, config=CFG, device=dev)
    bucket = torch.zeros(n, device=dev)
    residual = torch.zeros(n, device=dev)
    peers = [grad(n, torch.float32, 1500 + r, dev) for r in range(world)]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):                      # warm up on a side stream, as graph capture requires
        plan.quantize_chunks(bucket, residual=residual, new_residual=residual)
        plan.reduce_received(op="mean")
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        plan.quantize_chunks(bucket, residual=residual, new_residual=residual)
        plan.reduce_received(op="mean")
    cpu_residual = torch.zeros(n)
    shard = n // world
    for step in range(4):                              # replays interleaved with eager work and synchronisation
        g = grad(n, torch.float32, 1600 + step, dev)
        bucket.copy_(g)
        for src in range(world):                        # synthetic exchange: peers' chunk 0 payloads
            row = plan.received[src, :plan.payload_bytes]
            assert ops.quant_pack_payload_into(peers[src][:shard] * (1.0 + 0.01 * step), row)
        if step == 0:
            residual.zero_()
        graph.replay()
        torch.cuda.synchronize()
        prepared = g.cpu() + cpu_residual
        want_rows = [codec_torch.quantize(prepared[d * shard:(d + 1) * shard]) for d in range(world)]
        for d in range(world):
            assert torch.equal(plan.send[d, :plan.payload_bytes].cpu(), codec_torch.pack(*want_rows[d])), (step, d)
        cpu_residual = prepared - torch.cat([codec_torch.dequantize(c, s, shard) for c, s in want_rows])
        assert same_bits(residual, cpu_residual), step
        received = [codec_torch.quantize(peers[src][:shard].cpu() * (1.0 + 0.01 * step)) for src in range(world)]
        assert same_bits(plan.shard, codec_torch.reduce_payloads(received, shard, 64, "fp32", "mean")), step


@pytest.mark.parametrize("wire_format", ["portable", "native", "reduce_scatter", "reduce_scatter_pipelined"])
def test_hook_on_a_real_distributed_data_parallel_model(hip_device, wire_format):
    """register_comm_hook on torch's own DDP (one rank, RCCL): real GradBucket objects and futures, gradients within
    the quantization error of the uncompressed model.  Runs in a child process under a time limit so that trouble in
    process-group set-up cannot stall the test run."""
    import json
    import subprocess
    import sys
    from pathlib import Path

    worker = Path(__file__).resolve().parent / "workers" / "ddp_single_rank.py"
    done = subprocess.run([sys.executable, str(worker), wire_format], capture_output=True, text=True, timeout=240)
    assert done.returncode == 0, done.stderr[-2000:]
    report = json.loads([line for line in done.stdout.splitlines() if line.startswith("{")][-1])
    assert report["finite"] and report["buckets"] >= 3
    assert all(0.0 < e < 0.02 for e in report["errors"]), report
    if wire_format == "reduce_scatter_pipelined":       # three iterations: flushed after each one's last bucket
        assert report["pipeline"]["flushes"] == 3 and report["pipeline"]["pending"] == 0, report
        assert report["pipeline"]["buckets"] == report["buckets"]
