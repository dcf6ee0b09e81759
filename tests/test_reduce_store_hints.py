"""How the fused reduce stores outputs that no descriptor covers - tensors at element alignment and a tensor's last block - read off the
compiled kernels: non-temporal wherever the policy of whole blocks has that hint, whatever else it has beside it."""
import re
import subprocess
from pathlib import Path

CSRC = Path(__file__).resolve().parents[1] / "lowbit_comm_amd" / "csrc"
PROBE = """
#include "dequant_reduce_block.h"
namespace lbc {
template <typename OT, int W> __device__ void body(const ReduceArgs &a) { reduce::dequant_reduce_block<OT, 64, W, kUnaligned>(a, blockIdx.x, gridDim.x); }
#define KERNEL(name, OT, W) extern "C" __global__ __launch_bounds__(kBlock) void name(const ReduceArgs a) { body<OT, W>(a); }
%s
}  // namespace lbc
"""
# (element type, payloads) -> whether the outputs leave non-temporal: they do unless the reads outweigh the writes by 1.6 and more
CASES = {("float", 2): True, ("float", 4): True, ("float", 8): False, ("bf16", 1): True, ("bf16", 2): True, ("f16", 2): True,
         ("bf16", 4): False, ("f16", 8): False}


def test_stores_without_a_descriptor_keep_the_non_temporal_hint(tmp_path):
    makefile = (CSRC / "Makefile").read_text()
    flags = re.search(r"HIPFLAGS\s*:=\s*((?:.*\\\n)*.*)", makefile).group(1).replace("\\\n", " ").split()
    flags = [f.replace("$(ARCH)", "gfx950") for f in flags if f != "-fPIC"]
    source, listing = tmp_path / "probe.hip", tmp_path / "probe.s"
    source.write_text(PROBE % "\n".join(f"KERNEL(k_{t}_{w}, {t}, {w})" for t, w in CASES))
    subprocess.run(["/opt/rocm/bin/hipcc", *flags, "-I", str(CSRC), "--cuda-device-only", "-S", str(source), "-o", str(listing)],
                   check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL, timeout=600)
    text = listing.read_text()
    for (name, world), hinted in CASES.items():
        body = text[text.index(f"\nk_{name}_{world}:"):]
        body = body[:body.index("s_endpgm")]
        # whole vectors; the one that the tensor's end cuts short leaves element by element, without a hint
        stores = re.findall(r"^\s*(?:global|flat)_store_dwordx4 [^\n]*", body, flags=re.M)
        assert stores and all(line.rstrip().endswith(" nt") == hinted for line in stores), (name, world, stores)
