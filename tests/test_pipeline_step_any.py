"""The shared grid for buckets at element alignment and groups of 32 and 16 (lbc_bucket_pipeline_step_any): every byte equals what
the separate launches write, and the pipelined transport uses it for buckets of any size."""
import numpy as np
import pytest
import torch

from lowbit_comm_amd import CompressionConfig

pytestmark = pytest.mark.gpu
TYPES = (torch.float32, torch.bfloat16, torch.float16)


@pytest.fixture(scope="module")
def ops(hip_device):
    from lowbit_comm_amd.hip import ops

    return ops


def gradient(n, dtype, seed, dev, sigma=1e-3):
    return (torch.randn(n, generator=torch.Generator().manual_seed(seed)) * sigma).to(dtype).to(dev)


# chunk sizes at the edges of tiles and blocks of 4 and 8 elements a lane, one element, remainders, whole groups, and odd
# starts (`shift` elements off a 16-byte line)
@pytest.mark.parametrize("group", (64, 32, 16))
@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("with_residual", (False, True))
def test_any_layout_equals_the_separate_launches(ops, hip_device, group, dtype, with_residual):
    rng = np.random.default_rng(group + 7 * TYPES.index(dtype) + with_residual)
    sizes = [1, 15, 63, 64, 65, 255, 257, 1023, 1025, 2049, 4095, 4097, 8191, 12_289]
    for case, (shard, world) in enumerate((s, int(rng.integers(1, 9))) for s in sizes):
        n = max(1, shard * world - int(rng.integers(0, min(world, shard))))          # the last chunk may be short
        shard = -(-n // world)
        shift = case % 3
        what = f"group {group} {dtype} n {n} world {world} shift {shift} residual {with_residual}"
        nbytes = ops.payload_nbytes(shard, group)
        stride = -(-nbytes // 256) * 256
        x = gradient(n + shift, dtype, 10 + case, hip_device)[shift:]
        residual = gradient(n + shift, torch.float32, 20 + case, hip_device, 1e-5)[shift:] if with_residual else None
        keep = None if residual is None else residual.clone()
        send = torch.zeros(world, stride, dtype=torch.uint8, device=hip_device)
        received, gathered = (torch.zeros(world, stride, dtype=torch.uint8, device=hip_device) for _ in range(2))
        for r in range(world):
            for rows, seed in ((received, 100), (gathered, 200)):
                assert ops.quant_pack_payload_into(gradient(shard, dtype, seed + r, hip_device), rows[r, :nbytes], group_size=group)
        mine = torch.zeros(nbytes, dtype=torch.uint8, device=hip_device)
        out = torch.zeros(n + shift, dtype=dtype, device=hip_device)
        quant = ops.bind_quant_pack_chunks(x, send, world, group_size=group, residual=residual, new_residual=residual)
        pairs = [ops.split_payload(received[r, :nbytes], shard, group) for r in range(world)]
        reduce = ops.bind_dequant_reduce_quant(pairs, *ops.split_payload(mine, shard, group), shard, group_size=group,
                                               divisor=float(world), mid_dtype=dtype)
        decode = ops.bind_dequant_chunks(gathered, out[shift:], shard, group_size=group)
        held = [t for t in (send, mine, out, residual) if t is not None]
        for stages in ("qrd", "qr", "qd", "rd"):
            outcome = []
            step = ops.bind_bucket_pipeline_step(*(launch if name in stages else None
                                                   for name, launch in zip("qrd", (quant, reduce, decode))), any_layout=True)
            for launches in ((step,), tuple(launch for name, launch in zip("qrd", (quant, reduce, decode)) if name in stages)):
                send.zero_(), mine.zero_(), out.zero_()
                if residual is not None:
                    residual.copy_(keep)
                for launch in launches:
                    assert launch() is True, f"{what} stages {stages}"
                outcome.append([t.clone() for t in held])
            for got, want in zip(*outcome):
                assert torch.equal(got.view(torch.uint8), want.view(torch.uint8)), f"{what} stages {stages}"


@pytest.mark.parametrize("group", (64, 32))
@pytest.mark.parametrize("error_feedback", (False, True))
def test_pipelined_transport_shares_launches_for_buckets_of_any_size(hip_device, group, error_feedback):
    from lowbit_comm_amd.hip.reduce_scatter import make_reduce_scatter_transport

    def all_to_all(received, send):
        received.copy_(send)

    def all_gather(gathered, mine):
        gathered[1:, :mine.numel()] = mine

    sizes, config = (70_001, 33_333, 64 * 8 * 40, 100_003), CompressionConfig(group_size=group)
    common = dict(world_size=8, rank=0, all_to_all=all_to_all, all_gather=all_gather, error_feedback=error_feedback)
    piped, plain = make_reduce_scatter_transport(pipelined=True, **common), make_reduce_scatter_transport(**common)
    mine = [gradient(n, torch.bfloat16, 300 + n, hip_device) for n in sizes]
    theirs = [t.clone() for t in mine]
    futures = [piped(t, config=config, op="mean") for t in mine]
    piped.flush()
    for future, tensor in zip(futures, theirs):
        assert torch.equal(future.wait().view(torch.int16), plain(tensor, config=config, op="mean").view(torch.int16))
    assert piped.pipeline.stats["merged_launches"] == len(sizes) and piped.pipeline.stats["separate_launches"] == 2


def test_any_layout_still_says_what_has_no_shared_grid(ops, hip_device):
    n, world = 64 * 4 * 9 + 3, 4
    shard = -(-n // world)
    send = torch.zeros(world, 1024, dtype=torch.uint8, device=hip_device)
    x = gradient(n, torch.bfloat16, 1, hip_device)
    half = gradient(n, torch.bfloat16, 2, hip_device, 1e-5)
    mine = torch.zeros(ops.payload_nbytes(shard), dtype=torch.uint8, device=hip_device)
    pairs = [ops.quant_pack(gradient(shard, torch.bfloat16, 3 + r, hip_device)) for r in range(world)]

    def reduce(kind):
        return ops.bind_dequant_reduce_quant(pairs, *ops.split_payload(mine, shard), shard, mid_dtype=kind)

    plain = ops.bind_quant_pack_chunks(x, send, world)
    assert ops.bind_bucket_pipeline_step(plain, reduce(torch.bfloat16), any_layout=True)() is True
    assert ops.bind_bucket_pipeline_step(plain, reduce(torch.bfloat16))() is False
    assert ops.bind_bucket_pipeline_step(plain, reduce(torch.float32), any_layout=True)() is False
    assert ops.bind_bucket_pipeline_step(ops.bind_quant_pack_chunks(x, send, world, residual=half), reduce(torch.bfloat16),
                                         any_layout=True)() is False


def test_native_step_stands_back_for_replaced_parts(hip_device, monkeypatch):
    """A plan whose method has been replaced (its class or the instance), a subclass of the pipeline and a merge step of its own
    are asked as before the native call; every way gives the same bucket."""
    from lowbit_comm_amd.hip import bucket_pipeline
    from lowbit_comm_amd.hip.reduce_scatter import ReduceScatterPlan

    def run(make=bucket_pipeline.BucketPipeline, prepare=None, **kwargs):
        pipe = make(world_size=4, rank=0, all_to_all=lambda received, send: received.copy_(send),
                    all_gather=lambda gathered, mine: gathered[1:, :mine.numel()].copy_(mine), **kwargs)
        tensors = [gradient(n, torch.bfloat16, n, hip_device) for n in (10_001, 10_001, 4096, 10_001)]
        for _ in range(2):
            if prepare is not None and pipe._plans:
                prepare(pipe)
            futures = [pipe.submit(t, config=CompressionConfig()) for t in tensors]
            pipe.flush()
        return [f.wait().clone() for f in futures]

    want = run()
    seen = []
    quantize, decode, requantize = (getattr(ReduceScatterPlan, "bound_" + n) for n in ("quantize", "decode", "reduce_requantize"))

    def on_instances(pipe):
        for plan in next(iter(pipe._plans.values())):
            plan.bound_decode = lambda *a, plan=plan, **k: seen.append("instance") or decode(plan, *a, **k)

    class Sub(bucket_pipeline.BucketPipeline):
        def _launch(self, *args):
            seen.append("subclass")
            return super()._launch(*args)

    outcomes = [run(prepare=on_instances), run(make=Sub),
                run(merge_stages=lambda q, r, d: seen.append("merge") or (lambda stream=None: False))]
    with monkeypatch.context() as patched:
        patched.setattr(ReduceScatterPlan, "bound_quantize", lambda self, *a, **k: seen.append("class") or quantize(self, *a, **k))
        outcomes.append(run())
    assert set(seen) == {"instance", "subclass", "merge", "class"}
    for outcome in outcomes:
        assert all(torch.equal(a.view(torch.int16), b.view(torch.int16)) for a, b in zip(outcome, want))


def test_native_step_leaves_other_operands_to_the_bound_launches(hip_device):
    """A strided bucket is refused as it was, an output of its own is taken; buffers that are no plan's are refused."""
    from lowbit_comm_amd import _host
    from lowbit_comm_amd.hip.bucket_pipeline import BucketPipeline

    def make():
        return BucketPipeline(world_size=2, rank=0, all_to_all=lambda received, send: received.copy_(send),
                              all_gather=lambda gathered, mine: gathered[1:, :mine.numel()].copy_(mine))

    base = gradient(2 * 6400, torch.float32, 5, hip_device)
    with pytest.raises(RuntimeError, match="contiguous"):
        make().submit(base[::2], config=CompressionConfig())
    pipe, out = make(), torch.empty(6400, device=hip_device)
    futures = [pipe.submit(base[:6400].clone(), config=CompressionConfig()),
               pipe.submit(base[:6400].clone(), config=CompressionConfig(), out=out)]
    pipe.flush()
    first, second = (f.wait() for f in futures)
    assert second.data_ptr() == out.data_ptr() and torch.equal(first, second)
    rows = torch.zeros(2, 64, dtype=torch.uint8, device=hip_device)
    with pytest.raises(ValueError, match="do not belong"):
        _host.Stages(6400, 2, 0, 64, 0, rows, rows, rows)


def step_kernels(run):
    """The shared-grid kernels that `run` launches, as (access mode, group size); fp32 buckets only."""
    import re

    from torch.profiler import ProfilerActivity, profile

    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        run()
        torch.cuda.synchronize()
    found = [re.search(r"bucket_pipeline_step_kernel<float, \w+, \d+, \d+, (\d+), (\d+)>", e.name) for e in prof.events()]
    return [tuple(int(v) for v in f.groups()) for f in found if f]


MODES = {"auto": 2, "stream": 2, "cached": 1}      # kStream, kVector


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("group", (64, 32, 16))
@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("error_feedback", (False, True))
def test_pipelined_transport_launches_in_the_default_access_mode(ops, hip_device, dtype, error_feedback, group, mode):
    from lowbit_comm_amd.hip.reduce_scatter import make_reduce_scatter_transport

    def run(transport, tensors):
        futures = [transport(t, config=CompressionConfig(group_size=group), op="mean") for t in tensors]
        transport.flush()
        return [f.wait() for f in futures]

    def transport(**kwargs):
        return make_reduce_scatter_transport(world_size=4, rank=0, all_to_all=lambda received, send: received.copy_(send),
                                             all_gather=lambda gathered, mine: gathered[1:, :mine.numel()].copy_(mine),
                                             error_feedback=error_feedback, **kwargs)

    sources = [gradient(64 * 4 * 40, dtype, 400 + k, hip_device) for k in range(4)]
    plain = transport()
    want = [plain(t.clone(), config=CompressionConfig(group_size=group), op="mean") for t in sources]
    mine, pipe = [t.clone() for t in sources], transport(pipelined=True)
    with ops.access_mode(mode):
        kernels = step_kernels(lambda: run(pipe, mine))
    assert dtype != torch.float32 or kernels == [(MODES[mode], group)] * 4
    assert pipe.pipeline.stats["merged_launches"] == 4
    assert all(torch.equal(a.view(torch.uint8), b.view(torch.uint8)) for a, b in zip(mine, want))


@pytest.mark.parametrize("change", ("row stride", "spaced rows", "own row"))
def test_pipelined_transport_takes_plans_with_matrices_of_their_own(hip_device, change):
    """A plan whose receive matrix has another row stride or rows that are not back to back, and one that requantizes into a row
    of its own (which is what the gather is handed), give the buckets that the plain plan gives."""
    from lowbit_comm_amd.hip.bucket_pipeline import BucketPipeline
    from lowbit_comm_amd.hip.reduce_scatter import ReduceScatterPlan

    def factory(*args, **kwargs):
        plan = ReduceScatterPlan(*args, **kwargs)
        world, stride = plan.received.shape
        if change == "row stride":
            plan.received = torch.zeros(world, stride + 256, dtype=torch.uint8, device=hip_device)
        elif change == "spaced rows":
            plan.received = torch.zeros(world, 2 * stride, dtype=torch.uint8, device=hip_device)[:, :stride]
        else:
            plan.my_row = torch.zeros(plan.payload_bytes, dtype=torch.uint8, device=hip_device)
        return plan

    def run(**kwargs):
        pipe = BucketPipeline(world_size=4, rank=1, all_to_all=lambda received, send: received[:, :send.shape[1]].copy_(send),
                              all_gather=lambda gathered, mine: gathered[:, :mine.numel()].copy_(mine.clone()), **kwargs)
        futures = [pipe.submit(gradient(n, torch.bfloat16, n, hip_device), config=CompressionConfig()) for n in (10_001, 4096, 10_001, 10_001)]
        pipe.flush()
        return [f.wait().clone() for f in futures]

    for got, want in zip(run(plan_factory=factory), run()):
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))
