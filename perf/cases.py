"""Workloads of the compressed gradient path, as a training program runs them through the public entry points.

Six paths, each over the sizes, element types and options it is used with:

``codec``    ``quantize_tensor`` then ``dequantize_tensor`` of one tensor, in the portable payload format or in the CUDA
             extension's (the latter with its code books, stochastic rounding and outlier channel)
``local``    ``FusedErrorFeedbackCodec.step``: a bucket's local round trip with error feedback
``gather``   the comm hook's ``all_gather`` strategy: compensate, quantize, reduce of every rank's payload, residual update
``scatter``  an iteration's buckets through the comm hook's ``reduce_scatter`` strategy over the pipelined transport
``plan``     one bucket through ``compressed_all_reduce_via_reduce_scatter`` and a ``ReduceScatterPlan`` of its shape
``ring``     one bucket through the comm hook's ``topology`` strategy over the pipelined ring

One GPU is one rank.  The collectives are injected callables, as the entry points want them; here they leave the peers'
payloads in a receive buffer the first time they meet it and nothing afterwards, so the link is not part of a pass.
Gradients are N(0, 1e-3) with 0.1 % outliers N(0, 1e-1), residuals N(0, 1e-5).
"""
import math

import torch

from lowbit_comm_amd import CompressionConfig, dequantize_tensor, quantize_tensor
from lowbit_comm_amd.communication.ddp_hook import create_ddp_comm_hook
from lowbit_comm_amd.communication.gather_reduce import GatheredPayloads
from lowbit_comm_amd.hip.codec import FusedErrorFeedbackCodec
from lowbit_comm_amd.hip.loader import load_hip_extension
from lowbit_comm_amd.hip.reduce_scatter import (ReduceScatterPlan, compressed_all_reduce_via_reduce_scatter,
                                                make_reduce_scatter_transport)
from lowbit_comm_amd.hip.ring import make_pipelined_ring_transport
from lowbit_comm_amd.quantization.error_feedback import ErrorFeedbackState

DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
BYTES = {"fp32": 4, "fp16": 2, "bf16": 2}
MiB = 1 << 20


def _case(path, numel, dtype, **options):
    """Every case names every option, so that two cases can be compared field by field."""
    base = {"path": path, "numel": numel, "dtype": dtype, "wire": "portable", "group_size": 64, "bit": 8, "topk": 0,
            "quant_type": "linear", "stochastic": False, "compact": False, "error_feedback": False, "world": 1,
            "buckets": 1}
    base.update(options)
    return base


def listed():
    cases = {
        # a small tensor on its own (biases, norms, the last layers of a small model): one launch each way, odd length
        "codec small": _case("codec", 10_007, "fp32"),
        # one 25 MiB bucket, the size DistributedDataParallel makes by default
        "codec 25MiB fp32": _case("codec", 25 * MiB // 4, "fp32"),
        # the outlier channel of the CUDA extension's format, on a 50 MiB bucket of a mixed-precision run
        "codec outliers bf16": _case("codec", 25 * MiB, "bf16", wire="native", topk=2),
        # its 4-bit normal code book, the strongest compression on offer, interleaved scales
        "codec 4-bit normal fp32": _case("codec", 26_214_400, "fp32", wire="native", bit=4, quant_type="normal", compact=True),
        # the local error-feedback step on a 100 MiB mixed-precision bucket with an fp32 residual
        "local 100MiB bf16": _case("local", 50 * MiB, "bf16", error_feedback=True),
        # the comm hook's all_gather strategy with error feedback, eight ranks, default bucket
        "gather 25MiB bf16": _case("gather", 25 * MiB // 2, "bf16", error_feedback=True, world=8),
        # the same among ranks that run the CUDA extension, whose payloads are read and written as they are; fp32 training
        "gather native fp32": _case("gather", 25 * MiB // 4, "fp32", wire="native", error_feedback=True, world=8),
        # the first bucket of every DistributedDataParallel iteration is 1 MiB: a short iteration of such buckets
        "scatter 1MiB bf16": _case("scatter", MiB // 2, "bf16", world=8, buckets=4),
        # an iteration of sixteen default buckets with error feedback, eight ranks
        "scatter 16x25MiB bf16": _case("scatter", 25 * MiB // 2, "bf16", error_feedback=True, world=8, buckets=16),
        # the whole reduce-scatter + all-gather plan of a large fp32 bucket
        "plan 200MiB fp32": _case("plan", 50 * MiB, "fp32", world=8),
        # the same plan on a bucket whose parameters do not add up to a multiple of anything
        "plan odd bf16": _case("plan", 9_830_417, "bf16", world=8),
        # fourteen hops of the quantized ring on a default bucket
        "ring 25MiB bf16": _case("ring", 25 * MiB // 2, "bf16", world=8),
    }
    return [dict(case, name=name) for name, case in cases.items()]


def _size(rng, low, high, multiple=1):
    """Spread over the logarithm; half of the sizes as they fall (odd ones among them), half in whole KiB of elements."""
    n = int(math.exp(rng.uniform(math.log(low), math.log(high))))
    step = multiple if rng.random() < 0.5 else 1024
    return max(step, n // step * step)


def draw(rng):
    path = rng.choice(["codec", "codec native", "local", "gather", "gather native", "scatter", "plan", "ring"])
    dtype = rng.choice(["fp32", "bf16", "bf16", "fp16"])
    group = rng.choice([64, 64, 64, 32, 16])
    world = rng.choice([2, 4, 8, 8])
    if path == "codec":
        return _case("codec", _size(rng, 1_000, 50 * MiB), dtype, group_size=group)
    if path == "codec native":
        quant_type = rng.choice(["linear", "linear", "normal", "uniform", "e3m0", "e2m1"])
        bit = rng.choice([4, 8]) if quant_type == "linear" else 4
        return _case("codec", _size(rng, 1_000, 25 * MiB, multiple=64), dtype, wire="native", group_size=group, bit=bit,
                     quant_type=quant_type, topk=rng.choice([0, 1, 2]), stochastic=rng.random() < 0.4,
                     compact=rng.random() < 0.5)
    if path == "local":
        return _case("local", _size(rng, 10_000, 50 * MiB), dtype, group_size=group, error_feedback=True)
    if path == "gather":
        return _case("gather", _size(rng, 50_000, 25 * MiB), dtype, group_size=group, error_feedback=rng.random() < 0.7,
                     world=world)
    if path == "gather native":
        return _case("gather", _size(rng, 50_000, 25 * MiB, multiple=64), dtype, wire="native",
                     compact=rng.random() < 0.5, error_feedback=rng.random() < 0.7, world=world)
    if path == "scatter":
        return _case("scatter", _size(rng, 50_000, 25 * MiB // 2), dtype, group_size=rng.choice([64, 64, 32]),
                     error_feedback=rng.random() < 0.5, world=world, buckets=rng.randint(2, 12))
    if path == "plan":
        return _case("plan", _size(rng, 50_000, 50 * MiB), dtype, group_size=group, world=world)
    return _case("ring", _size(rng, 100_000, 25 * MiB), dtype, group_size=group, world=world)


# ---- inputs ------------------------------------------------------------------------------------
def _config(case):
    return CompressionConfig(bit=case["bit"], group_size=case["group_size"], topk=case["topk"],
                             quant_type=case["quant_type"], stochastic=case["stochastic"], compact=case["compact"],
                             error_feedback=case["error_feedback"], allow_experimental=case["bit"] != 8)


def _gradient(generator, numel, dtype):
    values = torch.randn(numel, device="cuda", generator=generator).mul_(1e-3)
    at = torch.randint(0, numel, (max(1, numel // 1000),), device="cuda", generator=generator)
    values[at] *= 100.0
    return values.to(dtype)


def _residual(generator, numel, dtype):
    return torch.randn(numel, device="cuda", generator=generator).mul_(1e-5).to(dtype)


class _Bucket:
    """What DistributedDataParallel hands to a comm hook."""

    def __init__(self, index, tensor, last):
        self._index, self._tensor, self._last = index, tensor, last

    def index(self):
        return self._index

    def buffer(self):
        return self._tensor

    def is_last(self):
        return self._last


def _rows(generator, case, numel, stride):
    """One payload per rank for a chunk of ``numel`` elements, in rows of ``stride`` bytes."""
    config = _config(case)
    rows = torch.zeros(case["world"], stride, dtype=torch.uint8, device="cuda")
    for row in rows:
        payload = quantize_tensor(_gradient(generator, numel, DTYPES[case["dtype"]]), config)
        row[:payload.numel()] = payload
    return rows


def _payload_bytes(case, numel):
    """Bytes of one payload: codes, and per group the scale (fp32 in the portable format, the tensor's type in the other)
    with the outlier channel's words behind it."""
    words = 1 if case["topk"] == 0 else case["topk"] + 2
    scale = 4 if case["wire"] == "portable" else BYTES[case["dtype"]] * words
    return -(-numel // case["group_size"]) * (case["group_size"] * case["bit"] // 8 + scale)


def prepare(case, seed):
    generator = torch.Generator(device="cuda")
    generator.manual_seed(seed)
    torch.cuda.manual_seed(seed)                  # the stream that stochastic rounding draws from
    numel, dtype, world = case["numel"], DTYPES[case["dtype"]], case["world"]
    config = _config(case)
    state = {"path": case["path"], "config": config, "dtype": case["dtype"]}

    if case["path"] == "codec":
        state["status"] = load_hip_extension(wire_format=case["wire"])
        state["tensor"] = _gradient(generator, numel, dtype)

    elif case["path"] == "local":
        state["tensor"] = _gradient(generator, numel, dtype)
        state["feedback"] = ErrorFeedbackState({0: _residual(generator, numel, torch.float32)})
        state["codec"] = FusedErrorFeedbackCodec(config, error_feedback=state["feedback"])

    elif case["path"] == "gather":
        status = load_hip_extension(wire_format=case["wire"])
        bucket = _gradient(generator, numel, dtype)
        peers = [quantize_tensor(_gradient(generator, numel, dtype), config, extension_status=status)
                 for _ in range(world - 1)]
        feedback = ErrorFeedbackState({0: _residual(generator, numel, dtype)}) if case["error_feedback"] else ErrorFeedbackState()

        def all_gather(local):
            state["sent"] = local.buffer
            return GatheredPayloads([local.buffer] + peers, world)

        state.update(feedback=feedback, bucket=_Bucket(0, bucket, True),
                     hook=create_ddp_comm_hook(config, strategy="all_gather", reduce="mean", all_gather=all_gather,
                                               error_feedback=feedback, extension_status=status))

    elif case["path"] == "scatter":
        shard = -(-numel // world)
        nbytes = _payload_bytes(case, shard)
        peers = _rows(generator, case, shard, nbytes)
        state["sent"] = {}

        def all_to_all(received, send):
            if received.data_ptr() not in state["sent"]:
                received[:, :nbytes] = peers
                send[:, nbytes:] = 0
                state["sent"][received.data_ptr()] = send

        filled = set()

        def all_gather(gathered, mine):
            if gathered.data_ptr() not in filled:
                gathered[1:, :nbytes] = peers[1:]
                filled.add(gathered.data_ptr())

        transport = make_reduce_scatter_transport(world_size=world, rank=0, all_to_all=all_to_all, all_gather=all_gather,
                                                  error_feedback=case["error_feedback"], pipelined=True)
        count = case["buckets"]
        state.update(transport=transport,
                     buckets=[_Bucket(i, _gradient(generator, numel, dtype), i == count - 1) for i in range(count)],
                     hook=create_ddp_comm_hook(config, strategy="reduce_scatter", reduce="mean",
                                               reduce_scatter_all_gather=transport))

    elif case["path"] == "plan":
        plan = ReduceScatterPlan(numel, dtype, world_size=world, rank=0, config=config, device="cuda")
        plan.send.zero_()
        plan.received.copy_(_rows(generator, case, plan.chunks.shard_numel, plan.row_stride))
        plan.gathered.copy_(_rows(generator, case, plan.chunks.shard_numel, plan.row_stride))
        state.update(plan=plan, tensor=_gradient(generator, numel, dtype), world=world,
                     out=torch.empty(numel, dtype=dtype, device="cuda"))

    elif case["path"] == "ring":
        shard = -(-numel // world)
        arrived = {}
        for size in {shard, numel - (world - 1) * shard}:
            payload = quantize_tensor(_gradient(generator, size, dtype), config)
            arrived[payload.numel()] = payload
        filled, state["sent"] = set(), []

        class Done:
            def query(self):
                return True

            def wait_stream(self, stream):
                return None

        done = Done()

        def exchange(payload, received, *, send_peer, recv_peer, stream):
            if received.data_ptr() not in filled:
                with torch.cuda.stream(stream):
                    received.copy_(arrived[received.numel()])
                filled.add(received.data_ptr())
            state["sent"].append(payload)
            return done

        transport = make_pipelined_ring_transport(world_size=world, rank=0, exchange=exchange)
        state.update(bucket=_Bucket(0, _gradient(generator, numel, dtype), True),
                     hook=create_ddp_comm_hook(config, strategy="topology", reduce="mean", topology_all_reduce=transport))
    return state


# ---- one pass ----------------------------------------------------------------------------------
def run(state):
    path, config = state["path"], state["config"]
    if path == "codec":
        tensor, status = state["tensor"], state["status"]
        payload = quantize_tensor(tensor, config, extension_status=status)
        return payload, dequantize_tensor(payload, tensor.shape, config, dtype=state["dtype"], extension_status=status)
    if path == "local":
        payload, restored = state["codec"].step(0, state["tensor"])
        return payload.packed, restored, state["feedback"].get(0)
    if path == "gather":
        reduced = state["hook"](None, state["bucket"]).wait()
        return state["sent"], reduced, state["feedback"].get(0)
    if path == "scatter":
        hook = state["hook"]
        futures = [hook(None, bucket) for bucket in state["buckets"]]
        reduced = [future.wait() for future in futures]
        return reduced, list(state["sent"].values()), list(state["transport"].residuals.values())
    if path == "plan":
        plan = state["plan"]
        reduced = compressed_all_reduce_via_reduce_scatter(
            state["tensor"], config=config, world_size=state["world"], rank=0, all_to_all=lambda received, send: None,
            all_gather=lambda gathered, mine: None, op="mean", plan=plan, out=state["out"])
        return reduced, plan.send, plan.gathered
    state["sent"].clear()
    return state["hook"](None, state["bucket"]).wait(), list(state["sent"])


# ---- what a pass cannot do without -------------------------------------------------------------
def work(case):
    """Inputs read once, outputs written once; a payload that one launch writes and another reads counts once each way."""
    n, item, world = case["numel"], BYTES[case["dtype"]], case["world"]
    tensor = n * item
    shard = -(-n // world)
    payload = _payload_bytes(case, n)
    piece = _payload_bytes(case, shard)
    if case["path"] == "codec":
        total, flops = 2 * (tensor + payload), 6 * n
    elif case["path"] == "local":
        # gradient and fp32 residual in; payload, restored gradient and residual out
        total, flops = tensor + 4 * n + payload + tensor + 4 * n, 8 * n
    elif case["path"] == "gather":
        # bucket in, own payload out, every payload in, reduced bucket out; with feedback the residual in and out
        total = tensor + payload + world * payload + tensor + (2 * tensor if case["error_feedback"] else 0)
        flops = (4 + 2 * world) * n
    elif case["path"] in ("scatter", "plan"):
        # bucket in, chunks out; arrived chunks in, own shard's payload out; every shard's payload in, bucket out
        total = tensor + world * piece + world * piece + piece + world * piece + tensor
        total += 8 * n if case["error_feedback"] else 0
        flops = 8 * n
    else:
        # first chunk's quantize; per accumulating hop payload and chunk in, chunk and payload out; per gather hop payload
        # in, chunk out, payload on (none behind the last)
        chunk = shard * item
        total = chunk + piece + (world - 1) * (2 * piece + 2 * chunk) + (world - 1) * (2 * piece + chunk) - piece
        flops = 8 * n
    return {"bytes": total * case["buckets"], "flops": flops * case["buckets"]}


def tolerance(case):
    """The payload formats are fixed to the bit, and so is the order of every sum: payloads are exchanged with other
    implementations and every rank has to end with the same tensor."""
    return "exact"
