"""Outputs on both sides of the sizes, alignments and payload counts where the CUDA-format reduce and the decodes of either format
change how whole blocks store them: the same values as the general path of small calls, bit for bit."""
import pytest
import torch

from lowbit_comm_amd import CompressionConfig, dequantize_tensor, quantize_tensor
from lowbit_comm_amd.hip.loader import load_hip_extension

pytestmark = pytest.mark.gpu
MiB = 1 << 20


def _payload(numel, dtype, config, status, seed, device):
    generator = torch.Generator(device=device).manual_seed(seed)
    values = (torch.randn(numel, generator=generator, device=device) * 1e-3).to(dtype)
    return quantize_tensor(values, config, extension_status=status)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("wire", ["portable", "native"])
def test_decode_around_the_line(hip_device, dtype, wire):
    """A large decode against the decodes of its pieces, which stay below the line (pieces of whole blocks keep their scales)."""
    status, config = load_hip_extension(wire_format=wire), CompressionConfig()
    name, item = {torch.float32: ("fp32", 4), torch.bfloat16: ("bf16", 2)}[dtype]
    line = (32 if item == 4 else 20 if wire == "portable" else 16) * MiB // item
    for numel in sorted({start + step for start in (16 * MiB // item, line) for step in (-64, 0, 64 * 33)}):
        generator = torch.Generator(device=hip_device).manual_seed(numel)
        values = (torch.randn(numel, generator=generator, device=hip_device) * 1e-3).to(dtype)
        got = dequantize_tensor(quantize_tensor(values, config, extension_status=status), (numel,), config, dtype=name,
                                extension_status=status)
        for start in range(0, numel, 2 * MiB):
            piece = values[start:start + 2 * MiB].clone()
            want = dequantize_tensor(quantize_tensor(piece, config, extension_status=status), tuple(piece.shape), config,
                                     dtype=name, extension_status=status)
            assert torch.equal(got[start:start + 2 * MiB].view(torch.uint8), want.view(torch.uint8)), (numel, start)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("world", [3, 4, 8])
@pytest.mark.parametrize("offset", [0, 1])
def test_cuda_format_reduce_with_feedback(hip_device, dtype, world, offset):
    """Aligned and odd outputs, payload counts on both sides of the rule, sizes on both sides of a block and of the rule's lines,
    against torch in the kernel's own arithmetic: a sum in fp32 of code * (scale / 127), times 1 / world, rounded once."""
    from lowbit_comm_amd.hip import cuda_wire

    config, status = CompressionConfig(), load_hip_extension(wire_format="native")
    name = {torch.float32: "fp32", torch.bfloat16: "bf16"}[dtype]
    item = torch.empty((), dtype=dtype).element_size()
    lines = [line // item + step for line in ((3 * MiB // 2, 9 * MiB, 32 * MiB) if item == 4 else (MiB // 4, 32 * MiB))
             for step in (-576, 0, 64)] + [48 * MiB // item - 64, 48 * MiB // item]
    sizes = [64 * 5, 4096, 4096 * 9 + 64 * 3] + (lines if world == 4 and offset == 0 else [])
    for numel in sizes:
        payloads = [_payload(numel, dtype, config, status, 10 * r + 1, hip_device) for r in range(world)]
        prepared = (torch.randn(numel, device=hip_device) * 1e-3).to(dtype)
        out = torch.zeros(numel + offset, dtype=dtype, device=hip_device)[offset:]
        residual = torch.zeros(numel + offset, dtype=dtype, device=hip_device)[offset:]
        assert cuda_wire.dequant_reduce_into(payloads, out, inv_divisor=float(torch.tensor(1.0) / world), compact=config.compact, prepared=prepared,
                                             new_residual=residual, fused_multiply_add=False)
        total = torch.zeros(numel, dtype=torch.float32, device=hip_device)
        for payload in payloads:
            total += _terms(payload, numel, dtype)
        total *= torch.tensor(1.0) / world
        assert torch.equal(out.view(torch.int32 if item == 4 else torch.int16), total.to(dtype).view(torch.int32 if item == 4 else torch.int16)), numel
        left = (prepared.float() - total).to(dtype)
        assert torch.equal(residual.view(torch.int32 if item == 4 else torch.int16), left.view(torch.int32 if item == 4 else torch.int16)), numel


def _terms(payload, numel, dtype):
    """code * (scale / 127) of every element of a payload with its scales behind the codes, in fp32."""
    codes = payload[:numel].view(torch.int8)
    scales = payload[numel:].view(dtype).float()
    width = torch.empty((), dtype=dtype).element_size()               # bytes are reversed inside a word of the element's size
    codes = codes.view(-1, width).flip(1).reshape(-1, 64).float()
    step = scales / torch.full_like(scales, 127.0)                    # a division: by a number, torch multiplies by its reciprocal
    return (codes * step[:, None]).reshape(-1)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("world", [1, 2, 3, 4, 8])
@pytest.mark.parametrize("offset", [0, 1])
def test_portable_reduce_with_and_without_feedback(hip_device, dtype, world, offset):
    """The kernels that load the sum early and those that load it late or not at all, on both sides of a block's end and of the line of
    three fp32 payloads, against the oracle's fold."""
    from lowbit_comm_amd.hip import ops
    from oracle import codec_torch

    name, item = {torch.float32: ("fp32", 4), torch.bfloat16: ("bf16", 2)}[dtype]
    bits = torch.int32 if item == 4 else torch.int16
    block = 256 * 16 // item
    sizes = [1, 63, block - 1, block, 2 * block, 2 * block + 65, 9 * block + 3]
    sizes += [13 * MiB // 8 + step for step in (-1, 0)] if world == 3 and item == 4 and offset == 0 else []
    for numel in sizes:
        generator = torch.Generator().manual_seed(numel + world)
        payloads = [codec_torch.quantize((torch.randn(numel, generator=generator) * 1e-3).to(dtype), 64) for _ in range(world)]
        on_device = [(codes.to(hip_device), scales.to(hip_device)) for codes, scales in payloads]
        want = codec_torch.reduce_payloads(payloads, numel, 64, name, "mean")
        prepared = (torch.randn(numel, generator=generator) * 1e-3).to(dtype)
        for feedback in (False, True):
            out = torch.zeros(numel + offset, dtype=dtype, device=hip_device)
            residual = torch.zeros(numel + offset, dtype=dtype, device=hip_device)
            how = dict(prepared=prepared.to(hip_device), new_residual=residual[offset:]) if feedback else {}
            assert ops.dequant_reduce_into(on_device, out[offset:], group_size=64, divisor=float(world), **how)
            assert torch.equal(out[offset:].cpu().view(bits), want.view(bits)), (numel, feedback)
            if feedback:
                left = (prepared.float() - want.float()).to(dtype)
                assert torch.equal(residual[offset:].cpu().view(bits), left.view(bits)), numel
