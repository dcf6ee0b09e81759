"""The ring transport's synchronous calls run on whichever stream is current, and its asynchronous ones on a stream of its own;
both leave what the executor on a stream of its own leaves."""
import pytest
import torch

from lowbit_comm_amd import CompressionConfig

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float32))
def test_ring_on_the_callers_stream(hip_device, dtype):
    from lowbit_comm_amd.hip.ring import make_pipelined_ring_executor, make_pipelined_ring_transport
    from lowbit_comm_amd.quantization.codec import quantize_tensor

    world, n, config = 4, 64 * 4 * 30 + 5, CompressionConfig()
    generator = torch.Generator().manual_seed(3)
    arrived = {}
    for size in {-(-n // world), n - (world - 1) * -(-n // world)}:
        payload = quantize_tensor((torch.randn(size, generator=generator) * 1e-3).to(dtype).to(hip_device), config)
        arrived[payload.numel()] = payload
    torch.cuda.synchronize()
    used = []

    class Done:
        def query(self):
            return True

        def wait(self):
            pass

        def wait_stream(self, stream):
            pass

    def exchange(payload, received, *, send_peer, recv_peer, stream):
        used.append(stream.cuda_stream)
        with torch.cuda.stream(stream):
            received.copy_(arrived[received.numel()])
        return Done()

    name = {torch.bfloat16: "bf16", torch.float32: "fp32"}[dtype]
    source = (torch.randn(n, generator=generator) * 1e-3).to(dtype).to(hip_device)
    want = source.clone()
    executor = make_pipelined_ring_executor(config=config, dtype=name, numel=n, world_size=world, rank=0, exchange=exchange,
                                            device=str(hip_device))
    executor.run(want).wait()
    torch.cuda.synchronize()
    transport = make_pipelined_ring_transport(world_size=world, rank=0, exchange=exchange)
    bucket = source.clone()
    default, side = torch.cuda.current_stream(), torch.cuda.Stream()
    for stream in (default, side, default, side, side):       # a plan per stream, replayed on it
        torch.cuda.synchronize()
        used.clear()
        with torch.cuda.stream(stream):
            bucket.copy_(source)
            got = transport(bucket, config=config, op="mean").clone()
        torch.cuda.synchronize()
        assert set(used) == {stream.cuda_stream}
        assert torch.equal(got.view(torch.uint8), want.view(torch.uint8))
    # a plan per stream, with buffers of its own: one plan for both would have two streams write the same buffers
    (synchronous,) = transport.executors.values()
    plans = synchronous._runtime.plans
    assert [key[2] for key in plans] == [default.cuda_stream, side.cuda_stream]
    buffers = [{value.data_ptr() for key, value in plan.items() if key[0] in ("send", "recv")} for plan in plans.values()]
    assert all(len(b) >= 2 * (world - 1) for b in buffers) and not buffers[0] & buffers[1]
    bucket.copy_(source)
    work = transport(bucket, config=config, op="mean", async_op=True)
    got = work.wait().clone()
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.uint8), want.view(torch.uint8))
    assert used[-1] not in (default.cuda_stream, side.cuda_stream) and len(transport.executors) == 2
