"""Groups whose maximum is within a factor of a few of the largest finite value: scales of 2^120, 2^121 and FLT_MAX / 127, whose exponent holds
a hundredth of its mantissas only.  Codes, scales and the decoded values against the oracle, bit for bit."""
import numpy as np
import pytest
import torch

from oracle import codec_torch

pytestmark = pytest.mark.gpu
FLT_MAX = float(np.finfo(np.float32).max)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("g", [64, 32, 16])
def test_groups_with_the_largest_scales(hip_device, dtype, g):
    from lowbit_comm_amd.hip import ops

    top = float(torch.finfo(dtype).max)
    generator = torch.Generator().manual_seed(g)
    line = 127.0 * 2.0 ** 121                                          # from here on a scale has the last exponent
    maxima = [top, float(torch.tensor(top, dtype=dtype)) * (1 - 2.0 ** -8), line, line * (1 - 2.0 ** -8), 2.0 ** 127, 127.0 * 2.0 ** 120, 3.376e38]
    maxima += (line + (FLT_MAX - line) * torch.rand(4096, generator=generator).double()).clamp(max=top).tolist()
    groups = (torch.rand(len(maxima), g, generator=generator).double() * 2 - 1) * torch.tensor(maxima).double()[:, None]
    ties = (torch.arange(g).double() - g // 2 + 0.5) * (torch.tensor(maxima).double()[:, None] / 127)
    x = torch.where(torch.rand(len(maxima), g, generator=generator) < 0.5, groups, ties)
    x[:, 0] = torch.tensor(maxima).double()
    x = x.clamp(-top, top).to(dtype).reshape(-1)
    assert torch.isfinite(x.float()).all()
    codes, scales = ops.quant_pack(x.to(hip_device), group_size=g)
    want_codes, want_scales = codec_torch.quantize(x, g)
    assert (want_scales >= 2.0 ** 121).sum() > 3000
    assert torch.equal(scales.cpu().view(torch.int32), want_scales.view(torch.int32))
    assert torch.equal(codes.cpu(), want_codes)
