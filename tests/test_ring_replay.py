"""The ring transport's later calls on a bucket replay the launches and exchanges of the first one without a submission around
them: the same bits, the same refusals, and the whole protocol where a caller has put something of its own in its place."""
import pytest
import torch

from lowbit_comm_amd import CompressionConfig
from lowbit_comm_amd.hip import ring

pytestmark = pytest.mark.gpu
CONFIG = CompressionConfig()


class Done:
    waited = 0

    def query(self):
        return True

    def wait(self):
        pass

    def wait_stream(self, stream):
        Done.waited += 1


def _ring(device, n=64 * 4 * 30 + 5, world=4, handle=Done, **options):
    from lowbit_comm_amd.hip.ring import make_pipelined_ring_transport
    from lowbit_comm_amd.quantization.codec import quantize_tensor

    generator = torch.Generator().manual_seed(5)
    arrived = {}
    for size in {-(-n // world), n - (world - 1) * -(-n // world)}:
        payload = quantize_tensor((torch.randn(size, generator=generator) * 1e-3).to(torch.bfloat16).to(device), CONFIG)
        arrived[payload.numel()] = payload
    state = {"fail": False, "handle": handle, "hops": 0}

    def exchange(payload, received, *, send_peer, recv_peer, stream):
        state["hops"] += 1
        if state["fail"] and state["hops"] % 6 == 4:
            raise OSError("link down")
        with torch.cuda.stream(stream):
            received.copy_(arrived[received.numel()])
        return state["handle"]()

    source = (torch.randn(n, generator=generator) * 1e-3).to(torch.bfloat16).to(device)
    return make_pipelined_ring_transport(world_size=world, rank=0, exchange=exchange, **options), source, state


def _same(a, b):
    return torch.equal(a.view(torch.int16), b.view(torch.int16))


def test_replays_give_the_first_calls_bits_and_wait_for_every_hop(hip_device, monkeypatch):
    transport, source, state = _ring(hip_device)
    bucket = source.clone()
    first = transport(bucket, config=CONFIG).clone()
    (executor,) = transport.executors.values()
    with monkeypatch.context() as patch:
        patch.setattr(ring, "_Submission", lambda **kw: pytest.fail("a replay makes no submission"))
        for _ in range(3):
            bucket.copy_(source)
            Done.waited = 0
            assert transport(bucket, config=CONFIG) is bucket and _same(bucket, first) and Done.waited == 6
    other = source.clone()                                    # another bucket has no record yet: the whole protocol
    assert _same(transport(other, config=CONFIG), first) and len(executor._runtime.plans) == 2


def test_a_failing_replay_is_held_like_a_failing_run_and_later_calls_work(hip_device):
    transport, source, state = _ring(hip_device)
    bucket = source.clone()
    first = transport(bucket, config=CONFIG).clone()
    (executor,) = transport.executors.values()
    state.update(fail=True, hops=0)
    with pytest.raises(OSError, match="link down"):
        transport(bucket, config=CONFIG)
    assert executor.pending_submission_count == 1
    state.update(fail=False, handle=object)
    with pytest.raises(AttributeError):                       # no wait_stream
        transport(bucket, config=CONFIG)

    class Blocking:
        def wait_stream(self, stream):
            pass

    state.update(handle=Blocking)
    with pytest.raises(TypeError, match="nonblocking query"):
        transport(bucket, config=CONFIG)
    state.update(handle=Done)
    torch.cuda.synchronize()
    bucket.copy_(source)
    assert _same(transport(bucket, config=CONFIG), first)
    for _ in range(2):                                        # a probe records its event the first time
        torch.cuda.synchronize()
        executor.reap_pending()
    assert executor.pending_submission_count == 0


def test_replaced_methods_managers_and_other_tensors_take_the_whole_protocol(hip_device):
    from lowbit_comm_amd.hip.completion import HipCompletionManager

    made = []

    class Manager(HipCompletionManager):
        def create_work(self, **kwargs):
            made.append(kwargs["result"])
            return super().create_work(**kwargs)

    transport, source, _ = _ring(hip_device, completion_manager=Manager())
    bucket = source.clone()
    first = transport(bucket, config=CONFIG).clone()
    for calls in (2, 3):
        bucket.copy_(source)
        assert _same(transport(bucket, config=CONFIG), first) and len(made) == calls
    transport, source, _ = _ring(hip_device)
    transport(bucket, config=CONFIG)
    (executor,) = transport.executors.values()
    runtime, seen = executor._runtime, []
    runtime.record_completion = lambda **kwargs: (seen.append(1), type(runtime).record_completion(runtime, **kwargs))[1]
    bucket.copy_(source)
    assert _same(transport(bucket, config=CONFIG), first) and seen == [1]
    del runtime.record_completion
    runs = []
    executor.run = lambda tensor: (runs.append(tensor), ring.PipelinedRingExecutor.run(executor, tensor))[1]
    for calls in (1, 2):                                      # an executor's own `run` sees every bucket, not the first alone
        bucket.copy_(source)
        assert _same(transport(bucket, config=CONFIG), first) and len(runs) == calls
    del executor.run
    wide = torch.zeros(source.numel() * 2, dtype=torch.bfloat16, device=hip_device)
    with pytest.raises(RuntimeError, match="contiguous"):
        transport(wide[::2], config=CONFIG)
