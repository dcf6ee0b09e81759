"""GPU parity where a lane's vector meets the end of a tensor or starts off a 16-byte line: sizes around the workgroups'
spans and the lanes' vectors, every start offset class, outputs inside guarded buffers that must keep their other bytes."""
import pytest
import torch

from oracle import codec_torch

pytestmark = pytest.mark.gpu

DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
GUARD = 37


def values(n, dtype, seed, sigma=1e-3):
    return (torch.randn(n, generator=torch.Generator().manual_seed(seed)) * sigma).to(dtype)


class Guarded:
    """`n` elements of `dtype` on the device, `offset` elements behind a pattern and with a pattern behind them."""

    def __init__(self, n, dtype, offset, device, fill=None):
        item = torch.empty((), dtype=dtype).element_size()
        self.backing = torch.full(((n + offset + GUARD) * item,), 0x5A, dtype=torch.uint8, device=device)
        self.inside = self.backing.view(dtype)[offset:offset + n]
        self.start, self.stop = offset * item, (offset + n) * item
        if fill is not None:
            self.inside.copy_(fill)

    def check(self, want, what):
        got = self.inside.cpu()
        assert torch.equal(got.view(torch.uint8), want.contiguous().view(torch.uint8)), what
        outside = torch.cat([self.backing[:self.start], self.backing[self.stop:]]).cpu()
        assert bool((outside == 0x5A).all()), f"{what}: wrote outside"


# a workgroup of the quantize spans 1024 elements (4 a lane) or 2048 (8 a lane) of a tensor that the chip holds at once
@pytest.mark.parametrize("n", [1, 5, 66, 1023, 1025, 2047, 2049, 4097, 8193, 2 * 8192 + 3])
@pytest.mark.parametrize("offset", [0, 1, 3])
@pytest.mark.parametrize("dtype", ["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("g", [64, 32, 16])
def test_quantize_at_block_ends_and_start_offsets(hip_device, g, dtype, offset, n):
    from lowbit_comm_amd.hip import ops

    t, world = DTYPES[dtype], 3
    for residual_type in (None, torch.float32):
        x = values(n, t, n + offset)
        r = None if residual_type is None else values(n, residual_type, n + 7, 1e-5)
        p = x if r is None else x + r
        shard = -(-n // world)
        x_in = Guarded(n, t, offset, hip_device, x)
        r_in = None if r is None else Guarded(n, residual_type, offset, hip_device, r)
        restored = Guarded(n, torch.float32, offset, hip_device)
        fresh = Guarded(n, torch.float32, offset, hip_device)
        prepared = Guarded(n, p.dtype, offset, hip_device)
        rows = torch.full((world, ops.payload_nbytes(shard, g) + 12), 0x5A, dtype=torch.uint8, device=hip_device)
        assert ops.quant_pack_chunks_into(x_in.inside, rows, world, group_size=g, residual=None if r is None else r_in.inside,
                                          new_residual=fresh.inside, restored=restored.inside, prepared_out=prepared.inside)
        padded = torch.zeros(world * shard, dtype=p.dtype)
        padded[:n] = p
        decoded = []
        for d in range(world):
            codes, scales = codec_torch.quantize(padded[d * shard:(d + 1) * shard], g)
            row, nbytes = rows[d].cpu(), ops.payload_nbytes(shard, g)
            assert torch.equal(row[:nbytes], codec_torch.pack(codes, scales)), (d, residual_type)
            assert bool((row[nbytes:] == 0x5A).all()), d
            decoded.append(codec_torch.dequantize(codes, scales, shard, g))
        want = torch.cat(decoded)[:n]
        restored.check(want, "restored")
        fresh.check(p.float() - want, "new residual")
        prepared.check(p, "prepared")
        x_in.check(x, "input")


# the tile count per wavefront changes where the chip holds no more: 2 Mi elements of four a lane, 4 Mi of eight
@pytest.mark.parametrize("dtype, residual_type, edge", [("fp32", None, 1 << 21), ("bf16", None, 1 << 22), ("bf16", "fp32", 1 << 21),
                                                        ("fp16", "fp16", 1 << 22)])
def test_quantize_on_both_sides_of_the_tile_rule(hip_device, dtype, residual_type, edge):
    from lowbit_comm_amd.hip import ops

    for n in (edge, edge + 1, edge + 4096 + 5):
        x = values(n, DTYPES[dtype], n)
        r = None if residual_type is None else values(n, DTYPES[residual_type], n + 7, 1e-5)
        p = x if r is None else x + r
        prepared = Guarded(n, p.dtype, 0, hip_device)
        payload = Guarded(ops.payload_nbytes(n), torch.uint8, 0, hip_device)
        assert ops.quant_pack_payload_into(x.to(hip_device), payload.inside, residual=None if r is None else r.to(hip_device),
                                           prepared_out=prepared.inside)
        payload.check(codec_torch.pack(*codec_torch.quantize(p)), f"payload of {n}")
        prepared.check(p, f"prepared of {n}")


def payloads_of(world, n, seed, device, g=64):
    """``world`` payloads covering ``n`` elements: (codes, scales) pairs for the oracle, packed tensors for the kernels."""
    pairs = [codec_torch.quantize(values(n, torch.float32, seed + r), g) for r in range(world)]
    return pairs, [codec_torch.pack(*pair).to(device) for pair in pairs]


# a workgroup of the decode spans 2048 (fp32) or 4096 (16-bit) outputs, of the reduce half of that from three payloads on
@pytest.mark.parametrize("n", [1, 7, 66, 1023, 2047, 2049, 4095, 4097, 4096 + 2048 + 5])
@pytest.mark.parametrize("offset", [0, 1, 3])
@pytest.mark.parametrize("dtype", ["fp32", "fp16", "bf16"])
def test_decode_and_reduce_at_block_ends_and_start_offsets(hip_device, dtype, offset, n):
    from lowbit_comm_amd.hip import ops

    t = DTYPES[dtype]
    pairs, packed = payloads_of(8, n, 100 + n, hip_device)
    for op in ("none", "sum", "max"):
        old = values(n, t, n + 1)
        out = Guarded(n, t, offset, hip_device, old)
        assert ops.dequant_payload_into(packed[0], out.inside, reduce_op=op)
        decoded = codec_torch.dequantize(*pairs[0], n, dtype=dtype)
        want = {"none": decoded, "sum": old + decoded, "max": torch.where(old > decoded, old, decoded)}[op]
        out.check(want, f"decode {op}")
    for world in (1, 2, 8):
        p = values(n, t, n + 2)
        out, fresh = Guarded(n, t, offset, hip_device), Guarded(n, t, offset, hip_device)
        prepared = Guarded(n, t, offset, hip_device, p)
        assert ops.dequant_reduce_into(packed[:world], out.inside, divisor=float(world), prepared=prepared.inside,
                                       new_residual=fresh.inside)
        want = codec_torch.reduce_payloads(pairs[:world], n, dtype=dtype, reduce="mean")
        out.check(want, f"reduce of {world}")
        fresh.check((p.float() - want.float()).to(t), f"residual of {world}")
    # shards of an odd bucket: every shard but the first starts off a 16-byte line
    world, shard = 3, -(-n // 3)
    shard_pairs, shard_packed = payloads_of(world, shard, 200 + n, hip_device)
    rows = torch.zeros(world, shard_packed[0].numel() + 4, dtype=torch.uint8, device=hip_device)
    for row, payload in zip(rows, shard_packed):
        row[:payload.numel()] = payload
    out = Guarded(n, t, offset, hip_device)
    assert ops.dequant_chunks_into(rows, out.inside, shard)
    out.check(torch.cat([codec_torch.dequantize(*pair, shard, dtype=dtype) for pair in shard_pairs])[:n], "shards")


# a workgroup of the ring step spans 1024 (fp32) or 2048 (16-bit) elements, 4096 of a 16-bit chunk above 4 Mi elements
@pytest.mark.parametrize("g, n", [(64, n) for n in (1, 7, 66, 1023, 1025, 2047, 2049, 4097, 8193, (1 << 22) + 4095, (1 << 22) + 4097)] +
                         [(g, n) for g in (32, 16) for n in (1, 7, 33, 66, 1023, 1025, 2049, 4097)])
@pytest.mark.parametrize("offset", [0, 1, 3])
@pytest.mark.parametrize("dtype", ["fp32", "fp16", "bf16"])
def test_ring_step_and_feedback_update_at_block_ends_and_start_offsets(hip_device, dtype, offset, g, n):
    from lowbit_comm_amd.hip import ops

    t = DTYPES[dtype]
    (pair,), (received,) = payloads_of(1, n, 300 + n, hip_device, g)
    start = values(n, t, n + 3)
    for op in ("sum", "none"):
        chunk = Guarded(n, t, offset, hip_device, start)
        send = Guarded(received.numel(), torch.uint8, 3 * offset, hip_device)
        scales_at = -(-n // g) * g
        if (send.inside.data_ptr() + scales_at) % 4 == 0:        # the payload's scales must lie on 4 bytes
            assert ops.ring_step_into(received, chunk.inside, send.inside, group_size=g, reduce_op=op, divisor=2.0)
        else:
            send = Guarded(received.numel(), torch.uint8, 0, hip_device)
            assert ops.ring_step_into(received, chunk.inside, send.inside, group_size=g, reduce_op=op, divisor=2.0)
        decoded = codec_torch.dequantize(*pair, n, g, dtype=dtype)
        want = (start + decoded if op == "sum" else decoded) / 2
        chunk.check(want, f"chunk {op}")
        send.check(codec_torch.pack(*codec_torch.quantize(want, g)), f"payload {op}")
    prepared, restored = values(n, t, n + 4), values(n, t, n + 5)
    residual = Guarded(n, t, offset, hip_device)
    assert ops.ef_update_into(Guarded(n, t, offset, hip_device, prepared).inside,
                              Guarded(n, t, offset, hip_device, restored).inside, residual.inside)
    residual.check((prepared.float() - restored.float()).to(t), "feedback update")


# codes of the reduce + requantize at byte addresses of every class, in and out; scales stay on 4 bytes
@pytest.mark.parametrize("g, n", [(g, n) for g in (64, 32, 16) for n in (1, 66, 1023, 1025, 2047, 2049, 8193)])
@pytest.mark.parametrize("offset", [1, 2, 3, 4])
@pytest.mark.parametrize("mid", ["fp32", "bf16"])
def test_reduce_requantize_of_codes_at_odd_addresses(hip_device, mid, offset, g, n):
    from lowbit_comm_amd.hip import ops

    for world in (1, 3, 8):
        pairs, _ = payloads_of(world, n, 400 + n, hip_device, g)
        held = [(Guarded(codes.numel(), torch.int8, offset + r % 2, hip_device, codes), scales.to(hip_device))
                for r, (codes, scales) in enumerate(pairs)]
        codes = Guarded(pairs[0][0].numel(), torch.int8, offset, hip_device)
        scales = Guarded(pairs[0][1].numel(), torch.float32, 1, hip_device)
        assert ops.dequant_reduce_quant_into([(c.inside, s) for c, s in held], codes.inside, scales.inside, n, group_size=g,
                                             divisor=float(world), mid_dtype=DTYPES[mid])
        reduced = codec_torch.reduce_payloads(pairs, n, g, mid, "mean")
        want_codes, want_scales = codec_torch.quantize(reduced, g)
        codes.check(want_codes, f"codes of {world}")
        scales.check(want_scales, f"scales of {world}")


# The CUDA byte format: a workgroup spans 1024 elements (fp32) or 2048 (16-bit) of a tensor that the chip holds at once,
# the reduce of up to two payloads and the decode twice that; a group's scale sits with its last lane
@pytest.mark.parametrize("n", [1, 60, 67, 131, 1023, 1025, 2047, 2049 + 64, 4095, 4097, 8192 + 3])
@pytest.mark.parametrize("compact", [True, False])
@pytest.mark.parametrize("dtype", ["fp32", "fp16", "bf16"])
def test_cuda_byte_format_at_block_ends(hip_device, dtype, compact, n):
    from lowbit_comm_amd.hip import cuda_wire
    from oracle import cuda_wire_np as wire
    from tests.test_cuda_wire_parity import from_numpy, to_numpy

    t = DTYPES[dtype]
    xs = [values(n, t, 10 * n + r) for r in range(3)]
    r = values(n, t, n + 7, 1e-5)
    payloads = []
    for x in xs:
        out = Guarded(cuda_wire.payload_nbytes(n, t), torch.uint8, 4, hip_device)
        assert cuda_wire.quant_pack_into(x.to(hip_device), out.inside, compact=compact)
        out.check(torch.from_numpy(wire.quantize(to_numpy(x), dtype, 64, compact)), "payload")
        payloads.append(out.inside.clone())
    out = Guarded(cuda_wire.payload_nbytes(n, t), torch.uint8, 4, hip_device)
    assert cuda_wire.quant_pack_into(xs[0].to(hip_device), out.inside, compact=compact, residual=r.to(hip_device))
    out.check(torch.from_numpy(wire.quantize(to_numpy(xs[0]), dtype, 64, compact, residual=to_numpy(r))), "payload with residual")
    host = [to_numpy(p) for p in payloads]
    old = values(n, t, n + 1)
    for op in ("none", "sum"):
        decoded = Guarded(n, t, 1, hip_device, old)
        assert cuda_wire.dequant_into(payloads[0], decoded.inside, compact=compact, reduce_op=op)
        decoded.check(from_numpy(wire.dequantize(host[0], n, dtype, 64, compact, op, to_numpy(old)), dtype, "cpu"), f"decode {op}")
    for world in (1, 2, 3):
        p = values(n, t, n + 2)
        reduced, fresh = Guarded(n, t, 1, hip_device), Guarded(n, t, 1, hip_device)
        assert cuda_wire.dequant_reduce_into(payloads[:world], reduced.inside, compact=compact, inv_divisor=1.0 / world,
                                             prepared=Guarded(n, t, 1, hip_device, p).inside, new_residual=fresh.inside)
        want, left = wire.reduce_mean_error_feedback(host[:world], to_numpy(p), n, dtype, divisor=world, compact=compact)
        reduced.check(from_numpy(want, dtype, "cpu"), f"reduce of {world}")
        fresh.check(from_numpy(left, dtype, "cpu"), f"residual of {world}")


# the tile count changes with the chip's wavefront slots: 2 Mi fp32 elements, 4 Mi and 8 Mi 16-bit ones
@pytest.mark.parametrize("dtype, with_residual, n", [("fp32", False, (1 << 21) + 5), ("fp32", True, (1 << 21) + 64),
                                                     ("bf16", False, (1 << 22) + 5), ("bf16", False, (1 << 23) + 64),
                                                     ("bf16", True, (1 << 22) + 64)])
def test_cuda_byte_format_beyond_the_tile_rule(hip_device, dtype, with_residual, n):
    from lowbit_comm_amd.hip import cuda_wire
    from oracle import cuda_wire_np as wire
    from tests.test_cuda_wire_parity import to_numpy

    t = DTYPES[dtype]
    x, r = values(n, t, n), values(n, t, n + 7, 1e-5) if with_residual else None
    out = Guarded(cuda_wire.payload_nbytes(n, t), torch.uint8, 4, hip_device)
    assert cuda_wire.quant_pack_into(x.to(hip_device), out.inside, residual=None if r is None else r.to(hip_device))
    out.check(torch.from_numpy(wire.quantize(to_numpy(x), dtype, 64, True, residual=None if r is None else to_numpy(r))), "payload")


# the sum of bucket and residual with its payload, against torch's add and the quantize of the padded sum: workgroup and
# lane ends, both sides of the tile rule (2 Mi fp32 elements, 4 Mi 16-bit ones), NaN and infinite elements
@pytest.mark.parametrize("n", [1, 5, 63, 64, 66, 1023, 1025, 2047, 2049, 8193, (1 << 21) + 5, (1 << 22) + 67])
@pytest.mark.parametrize("specials", [False, True])
@pytest.mark.parametrize("dtype", ["fp32", "fp16", "bf16"])
def test_compensated_quantize_of_the_cuda_byte_format(hip_device, dtype, specials, n):
    from lowbit_comm_amd import CompressionConfig, quantize_tensor
    from lowbit_comm_amd.hip.loader import load_hip_extension
    from lowbit_comm_amd.quantization.codec import compensate_and_quantize

    t, status = DTYPES[dtype], load_hip_extension(wire_format="native")
    x, r = values(n, t, n), values(n, t, n + 7, 1e-5)
    if specials:
        for seed, special in enumerate((float("nan"), float("inf"), float("-inf"))):
            for side, tensor in enumerate((x, r)):
                g = torch.Generator().manual_seed(100 * n + 10 * seed + side)
                tensor[torch.randint(0, n, (max(1, n // 300),), generator=g)] = special
    for offset, group, bit, compact in ((0, 64, 8, True), (1, 64, 8, False), (3, 64, 4, False), (0, 32, 4, True), (1, 16, 8, True)):
        config = CompressionConfig(bit=bit, group_size=group, compact=compact, allow_experimental=bit != 8)
        x_in, r_in = Guarded(n, t, offset, hip_device, x).inside, Guarded(n, t, offset, hip_device, r).inside
        want = x_in + r_in
        prepared, payload = compensate_and_quantize(x_in, r_in, config, extension_status=status)
        assert torch.equal(prepared.view(torch.uint8), want.view(torch.uint8)), "sum"
        assert torch.equal(payload, quantize_tensor(want, config, extension_status=status)), (group, bit, compact)


def test_compensated_quantize_leaves_other_operands_to_the_separate_calls(hip_device):
    from lowbit_comm_amd import CompressionConfig
    from lowbit_comm_amd.hip.loader import load_hip_extension
    from lowbit_comm_amd.quantization.codec import compensate_and_quantize

    status, config = load_hip_extension(wire_format="native"), CompressionConfig()
    x = torch.zeros(256, dtype=torch.bfloat16, device=hip_device)
    others = [x.float(), x[:128], x.view(4, 64), x.cpu(), torch.zeros(512, dtype=x.dtype, device=hip_device)[::2],
              x.clone().requires_grad_(True)]
    for other in others:
        assert compensate_and_quantize(x, other, config, extension_status=status) is None
        assert compensate_and_quantize(other, x, config, extension_status=status) is None
    assert compensate_and_quantize(x, x, CompressionConfig(topk=1), extension_status=status) is None
    assert compensate_and_quantize(x[:0], x[:0], config, extension_status=status) is None
    assert compensate_and_quantize(x, x, config, extension_status=load_hip_extension()) is None


@pytest.mark.parametrize("dtype, n", [("fp32", 100_001), ("bf16", 64 * 999)])
def test_hook_iterations_in_the_cuda_byte_format_match_the_separate_calls(hip_device, dtype, n):
    """A feedback state with a compensate step of its own takes the add and the quantize as two calls; both hooks keep the
    same residuals, payloads and results over several iterations."""
    from lowbit_comm_amd import CompressionConfig, quantize_tensor
    from lowbit_comm_amd.communication.ddp_hook import create_ddp_comm_hook
    from lowbit_comm_amd.communication.gather_reduce import GatheredPayloads
    from lowbit_comm_amd.hip.loader import load_hip_extension
    from lowbit_comm_amd.quantization.error_feedback import ErrorFeedbackState

    class OwnStep(ErrorFeedbackState):
        def compensate(self, key, tensor):
            return super().compensate(key, tensor)

    class Bucket:
        def __init__(self, tensor):
            self.tensor = tensor

        def index(self):
            return 0

        def buffer(self):
            return self.tensor

    t, status = DTYPES[dtype], load_hip_extension(wire_format="native")
    config = CompressionConfig(error_feedback=True)
    peer = quantize_tensor(values(n, t, 5).to(hip_device), config, extension_status=status)
    grads = [values(n, t, 20 + i).to(hip_device) for i in range(3)]
    seen = []
    for feedback in (ErrorFeedbackState(), OwnStep()):
        sent = []
        hook = create_ddp_comm_hook(config, strategy="all_gather", reduce="mean", error_feedback=feedback, extension_status=status,
                                    all_gather=lambda local: (sent.append(local.buffer), GatheredPayloads([local.buffer, peer], 2))[1])
        out = [hook(None, Bucket(g)).wait().clone() for g in grads]
        seen.append([*sent, *out, feedback.get(0)])
    for a, b in zip(*seen):
        assert torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8))


# a strided tensor that does not fill its last group is flattened on the way in; one of whole groups is refused
@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
@pytest.mark.parametrize("wire", ["portable", "native"])
def test_strided_ragged_tensors_quantize_like_their_flat_copies(hip_device, wire, dtype):
    from lowbit_comm_amd import CompressionConfig, quantize_tensor
    from lowbit_comm_amd.hip.loader import load_hip_extension

    status, config = load_hip_extension(wire_format=wire), CompressionConfig()
    x = values(70, DTYPES[dtype], 3).to(hip_device).view(7, 10).t()
    flat = torch.cat([x.reshape(-1), x.new_zeros(58)])
    assert torch.equal(quantize_tensor(x, config, extension_status=status), quantize_tensor(flat, config, extension_status=status))
    with pytest.raises(RuntimeError, match="contiguous"):
        quantize_tensor(flat.view(2, 64).t(), config, extension_status=status)


@pytest.mark.parametrize("divisor", [float("nan"), float("inf")])
def test_fused_reduce_of_the_cuda_byte_format_refuses_divisors_without_a_positive_reciprocal(hip_device, divisor):
    from lowbit_comm_amd import CompressionConfig, quantize_tensor
    from lowbit_comm_amd.hip.loader import load_hip_extension

    status = load_hip_extension(wire_format="native")
    module = status.module
    x = values(128, torch.float32, 5).to(hip_device)
    payload, out = quantize_tensor(x, CompressionConfig(), extension_status=status), torch.empty_like(x)
    policy = (64, 0, 8, module.QuantType.Linear, False)
    assert module.inplace_dequantize_reduce_mean([payload], out, *policy, 2.0)
    with pytest.raises(RuntimeError, match="divisor must be > 0"):
        module.inplace_dequantize_reduce_mean([payload], out, *policy, divisor)
    assert not module.inplace_dequantize_reduce_mean([payload], out[:100], *policy, divisor)   # not the fused reduce's


# whole tensors whose codes stay within reach of the decode: written through above 4 Mi fp32 elements, plain above 20 Mi 16-bit
# ones (16 Mi in the CUDA byte format); the last workgroup and the last group are cut short
@pytest.mark.parametrize("g", [64, 32, 16])
@pytest.mark.parametrize("dtype, n", [("fp32", (4 << 20) + 4096 + 5), ("fp16", (20 << 20) + 4096 + 5), ("bf16", (20 << 20) + 4096 + 5)])
def test_whole_tensors_whose_codes_are_kept(hip_device, dtype, n, g):
    from lowbit_comm_amd.hip import cuda_wire, ops
    from oracle import cuda_wire_np as wire
    from tests.test_cuda_wire_parity import to_numpy

    t = DTYPES[dtype]
    x = values(n, t, n + g)
    x_in = x.to(hip_device)
    out = Guarded(cuda_wire.payload_nbytes(n, t, g), torch.uint8, 4, hip_device)
    assert cuda_wire.quant_pack_into(x_in, out.inside, group_size=g, compact=False)
    out.check(torch.from_numpy(wire.quantize(to_numpy(x), dtype, g, False)), "payload of the CUDA byte format")
    out = Guarded(ops.payload_nbytes(n, g), torch.uint8, 16, hip_device)
    assert ops.quant_pack_payload_into(x_in, out.inside, group_size=g)
    out.check(codec_torch.pack(*codec_torch.quantize(x, g)), "portable payload")


def template_numbers(name):
    """The whole numbers among a kernel's template arguments, as the profiler prints them (mangled or not)."""
    import re

    if name.startswith("_Z"):
        return [int(v) for v in re.findall(r"Li(\d+)E", name)]
    return [int(v) for v in re.findall(r"(?<=[ <])\d+(?=[,>])", name)]


# which form the codes of a whole tensor are stored in: kStream 2 (non-temporal), kStreamThrough 3, kStreamKept 4
@pytest.mark.parametrize("dtype, new_residual, n, mode", [
    ("fp32", False, 4 << 20, 4), ("fp32", False, (4 << 20) + 64, 3), ("fp16", False, 20 << 20, 2), ("fp16", False, (20 << 20) + 64, 4),
    ("bf16", False, 20 << 20, 2), ("bf16", False, (20 << 20) + 64, 4), ("fp32", True, 10 << 20, 2), ("fp32", True, (10 << 20) + 64, 3),
    ("fp16", True, 10 << 20, 2), ("fp16", True, (10 << 20) + 64, 3)])
def test_store_form_of_a_whole_tensors_codes(hip_device, dtype, new_residual, n, mode):
    from lowbit_comm_amd.hip import ops
    from tests.test_zy_perf_gate import kernel_names

    x = torch.zeros(n, dtype=DTYPES[dtype], device=hip_device)
    payload = torch.empty(ops.payload_nbytes(n), dtype=torch.uint8, device=hip_device)
    fresh = torch.empty(n, device=hip_device) if new_residual else None
    (name,) = kernel_names(lambda: ops.quant_pack_payload_into(x, payload, new_residual=fresh))
    assert "quant_pack_kernel" in name and template_numbers(name)[:3] == [64, 4 if new_residual or dtype == "fp32" else 8, mode], name


# the same in the CUDA byte format, scales apart: 1 non-temporal, 0 plain, 2 written through
@pytest.mark.parametrize("dtype, n, codes", [("fp32", 4 << 20, 1), ("fp32", (4 << 20) + 64, 2), ("fp16", 16 << 20, 1),
                                             ("fp16", (16 << 20) + 64, 0), ("bf16", 16 << 20, 1), ("bf16", (16 << 20) + 64, 0)])
def test_store_form_of_a_whole_tensors_codes_in_the_cuda_byte_format(hip_device, dtype, n, codes):
    from lowbit_comm_amd.hip import cuda_wire
    from tests.test_zy_perf_gate import kernel_names

    x = torch.zeros(n, dtype=DTYPES[dtype], device=hip_device)
    payload = torch.empty(cuda_wire.payload_nbytes(n, x.dtype), dtype=torch.uint8, device=hip_device)
    (name,) = kernel_names(lambda: cuda_wire.quant_pack_into(x, payload, compact=False))
    assert "wire_quant_kernel" in name and template_numbers(name) == [64, 8, 1, codes, 4], name
