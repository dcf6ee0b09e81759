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


# a workgroup of the quantize spans 4096 (fp32) or 8192 (16-bit) elements, a lane 4 or 8
@pytest.mark.parametrize("n", [1, 5, 66, 4095, 4097, 8191, 8193, 2 * 8192 + 3])
@pytest.mark.parametrize("offset", [0, 1, 3])
@pytest.mark.parametrize("dtype", ["fp32", "fp16", "bf16"])
def test_quantize_at_block_ends_and_start_offsets(hip_device, dtype, offset, n):
    from lowbit_comm_amd.hip import ops

    t, world, g = DTYPES[dtype], 3, 64
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
        assert ops.quant_pack_chunks_into(x_in.inside, rows, world, residual=None if r is None else r_in.inside,
                                          new_residual=fresh.inside, restored=restored.inside, prepared_out=prepared.inside)
        padded = torch.zeros(world * shard, dtype=p.dtype)
        padded[:n] = p
        decoded = []
        for d in range(world):
            codes, scales = codec_torch.quantize(padded[d * shard:(d + 1) * shard], g)
            row, nbytes = rows[d].cpu(), ops.payload_nbytes(shard, g)
            assert torch.equal(row[:nbytes], codec_torch.pack(codes, scales)), (d, residual_type)
            assert bool((row[nbytes:] == 0x5A).all()), d
            decoded.append(codec_torch.dequantize(codes, scales, shard))
        want = torch.cat(decoded)[:n]
        restored.check(want, "restored")
        fresh.check(p.float() - want, "new residual")
        prepared.check(p, "prepared")
        x_in.check(x, "input")
