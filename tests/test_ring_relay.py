"""The hops of a ring that do not complete the sum: the payload of the updated chunk, and the chunk as it came."""
import ctypes

import numpy as np
import pytest
import torch

from lowbit_comm_amd import CompressionConfig
from lowbit_comm_amd.hip import library
from lowbit_comm_amd.hip.ring import HipPipelinedRingRuntime, RingSubmissionContext
from oracle import ring_np
from tests.test_ring_parity import DTYPES, tensor_like, to_np


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("g, offset", [(64, 0), (64, 1), (32, 0), (16, 3)])
def test_relay_writes_the_payload_of_the_sum_and_nothing_else(hip_device, dtype, g, offset):
    from lowbit_comm_amd.hip import ops

    block = 256 * 16 // DTYPES[dtype].itemsize                # elements one workgroup covers
    for seed, n in enumerate((1, g - 1, g, block - 1, block, block + g + 1, 5 * block + 3, 300_001)):
        received = torch.empty(ops.payload_nbytes(n, g), dtype=torch.uint8, device=hip_device)
        assert ops.quant_pack_payload_into(tensor_like(n, "fp32", seed, hip_device), received, group_size=g)
        backing = tensor_like(n + offset, dtype, 50 + seed, hip_device, sigma=3e-3)
        before, chunk = backing.clone(), backing[offset:]
        send = torch.full_like(received, 0xAB)
        assert ops.bind_ring_relay(received, chunk, send, group_size=g)()
        padded, raw = ops.num_groups(n, g) * g, received.cpu().numpy()
        _, (codes, scales) = ring_np.ring_step((raw[:padded].view(np.int8), raw[padded:].view(np.float32)), to_np(chunk, dtype),
                                               dtype, g, reduce_op="sum", divisor=1.0, emit=True)
        got = send.cpu().numpy()
        assert np.array_equal(got[:padded].view(np.int8), codes) and np.array_equal(got[padded:], scales.view(np.uint8)), n
        assert torch.equal(backing.view(torch.uint8), before.view(torch.uint8)), n


def test_relay_arguments_are_validated_before_any_device_work():
    lib, none, some = library.load_library(), ctypes.c_void_p(None), ctypes.c_void_p(64)
    assert lib.lbc_ring_relay(some, some, some, 0, 64, 64, none, none, 0, none) == -1
    assert "must not be null" in library.last_error(lib)
    assert lib.lbc_ring_relay(some, some, some, 0, -1, 64, some, some, 0, none) == -1
    assert lib.lbc_ring_relay(some, some, some, 7, 64, 64, some, some, 0, none) == -1
    assert lib.lbc_ring_relay(some, some, some, 0, 64, 64, some, some, 0, none) == -1       # send aliases the received payload
    assert lib.lbc_ring_relay(some, some, some, 0, 64, 48, some, some, 0, none) == 1
    assert lib.lbc_ring_relay(none, none, none, 0, 0, 64, none, none, 0, none) == 0


def test_a_runtime_with_steps_of_its_own_sees_every_updated_chunk():
    def context_of(runtime):
        context = RingSubmissionContext(tensor=None, stream=None, producer_completion=None)
        runtime.begin_schedule(context)
        return context.whole_schedule

    class Watching(HipPipelinedRingRuntime):
        def fused_reduce(self, *args, **kwargs):
            return super().fused_reduce(*args, **kwargs)

    common = dict(config=CompressionConfig(), dtype="fp32", world_size=4, rank=0, exchange=lambda *a, **k: None)
    assert context_of(HipPipelinedRingRuntime(**common))
    assert not context_of(Watching(**common)) and not context_of(HipPipelinedRingRuntime(fuse_steps=False, **common))
    replaced = HipPipelinedRingRuntime(**common)
    replaced.quant_pack = lambda *a, **k: None
    assert not context_of(replaced)
