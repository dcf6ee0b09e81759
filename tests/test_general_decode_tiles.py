"""The general decode of the CUDA byte format on both sides of the sizes where a wavefront takes two tiles, against the decodes of
the tensor's pieces, which are small enough for one: outliers and code books, whole and ragged last blocks, combining decodes."""
import pytest
import torch

pytestmark = pytest.mark.gpu
MiB = 1 << 20


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("bit, quant_type, topk", [(4, "normal", 0), (4, "e2m1", 1), (8, "linear", 2)])
@pytest.mark.parametrize("compact", [False, True])
def test_large_decodes_equal_the_decodes_of_their_pieces(hip_device, dtype, bit, quant_type, topk, compact):
    from lowbit_comm_amd.hip import cuda_wire

    policy = dict(group_size=64, bit=bit, quant_type=quant_type, topk=topk, compact=compact)
    line = (2 if dtype == torch.float32 else 4) * MiB
    generator = torch.Generator(device=hip_device).manual_seed(bit + topk)
    ends = (line, line + 64, line + 64 * 1031, 8 * MiB + 64)
    if dtype == torch.float32 and topk < 2:                   # two tiles up to 3 Mi elements, 4 Mi with an outlier
        ends += ((3 + topk) * MiB, (3 + topk) * MiB + 64)
    for numel in ends:
        x = (torch.randn(numel, generator=generator, device=hip_device) * 1e-3).to(dtype)
        base = (torch.randn(numel, generator=generator, device=hip_device) * 1e-3).to(dtype)

        def decoded(part, out, **how):
            payload = torch.empty(cuda_wire.general_payload_nbytes(part.numel(), dtype, 64, bit, topk), dtype=torch.uint8,
                                  device=hip_device)
            assert cuda_wire.bind_quant_general(part, payload, **policy)()
            assert cuda_wire.bind_dequant_general(payload, out, **policy, **how)()
            return out

        for how in ({}, {"reduce_op": "sum"}, {"reduce_op": "max"}, {"reduce_op": "min"}):
            got = decoded(x, base.clone(), **how)
            for start in range(0, numel, MiB):
                want = decoded(x[start:start + MiB].clone(), base[start:start + MiB].clone(), **how)
                assert torch.equal(got[start:start + MiB].view(torch.uint8), want.view(torch.uint8)), (numel, start, how)
