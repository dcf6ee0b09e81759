"""The topology transports keep executors between calls: what a call's policy is answered with does not depend on earlier calls."""
import pytest
import torch

from lowbit_comm_amd import CompressionConfig
from lowbit_comm_amd.hip.ring import HipPipelinedRingRuntime, make_pipelined_ring_transport
from lowbit_comm_amd.hip.tree import make_topology_transport

UNSERVED = (CompressionConfig(bit=4, allow_experimental=True), CompressionConfig(topk=2), CompressionConfig(quant_type="normal"))


@pytest.fixture(autouse=True)
def no_streams(monkeypatch):
    """A call gets as far as the look at the tensor's device, with or without a GPU."""
    monkeypatch.setattr(HipPipelinedRingRuntime, "_ready", lambda self: None)


def _ring():
    return make_pipelined_ring_transport(world_size=4, rank=0, exchange=lambda *a, **k: None)


def _topology():
    return make_topology_transport(world_size=4, rank=0, send=lambda *a, **k: None, recv=lambda *a, **k: None)


@pytest.mark.parametrize("make", [_ring, _topology])
@pytest.mark.parametrize("numel", [4 * 64 * 3, 4 * 64 * 3 + 5])      # the topology transport's ring and its tree
@pytest.mark.parametrize("config", UNSERVED)
def test_a_policy_without_kernels_is_refused_after_a_served_one_as_before_it(make, numel, config):
    transport, bucket = make(), torch.zeros(numel)
    with pytest.raises(ValueError, match="the ring runtime requires"):
        transport(bucket, config=config)
    assert not transport.executors
    with pytest.raises(RuntimeError, match="GPU tensor"):
        transport(bucket, config=CompressionConfig())
    assert len(transport.executors) == 1
    with pytest.raises(ValueError, match="the ring runtime requires"):
        transport(bucket, config=config)
    with pytest.raises(RuntimeError, match="GPU tensor"):
        transport(bucket, config=CompressionConfig(error_feedback=False, warmup_steps=3))
    assert len(transport.executors) == 1                              # fields that no executor reads share one


@pytest.mark.parametrize("change", [{"stochastic": True}, {"compact": True}, {"group_size": 32}])
def test_policies_that_an_executor_reads_have_executors_of_their_own(change):
    transport, bucket = _ring(), torch.zeros(4 * 64)
    for config in (CompressionConfig(), CompressionConfig(**change), CompressionConfig()):
        with pytest.raises(RuntimeError, match="GPU tensor"):
            transport(bucket, config=config)
    assert [e._runtime.config for e in transport.executors.values()] == [CompressionConfig(**change), CompressionConfig()]
