"""GPU parity of the one-launch input copies (solort_stage_inputs): the bytes of copy_ and fill_."""
from __future__ import annotations

import pytest
import torch

from solort_amd import ops

pytestmark = pytest.mark.gpu


# element counts at and around the 16-byte chunk and the 4 KB workgroup; none, one, two and three tensors
@pytest.mark.parametrize("sizes", [[], [1], [4, 3], [2048, 1, 5], [2047, 2049, 1024], [36 * 6144, 151936, 4]])
def test_stage_inputs(gpu, sizes):
    print(f"[stage_inputs {sizes}]", flush=True)
    dtypes = [torch.bfloat16, torch.float32, torch.int64]
    g = torch.Generator().manual_seed(len(sizes))
    srcs = [torch.randint(-9, 9, (n,), generator=g).to(dt).to(gpu) for n, dt in zip(sizes, dtypes)]
    bufs = [torch.full((s.numel() + 8,), 3, dtype=s.dtype, device=gpu) for s in srcs]
    pos = torch.zeros(1, dtype=torch.long, device=gpu)
    ops.stage_inputs([(b[: s.numel()], s) for b, s in zip(bufs, srcs)], pos, 1 << 40)
    assert pos.item() == 1 << 40
    for b, s in zip(bufs, srcs):
        assert torch.equal(b[: s.numel()], s) and (b[s.numel():] == 3).all()


def test_stage_inputs_other_forms(gpu):
    """What copy_ takes besides (other types, strides, devices, broadcasts) is still taken."""
    pos = torch.zeros(1, dtype=torch.long, device=gpu)
    want = torch.arange(64, dtype=torch.float32).view(8, 8)
    for src in (want.to(gpu, torch.bfloat16), want, want.t().contiguous().t().to(gpu), want[:1].to(gpu),
                torch.cat([torch.zeros(1), want.view(-1)]).to(gpu)[1:].view(8, 8)):
        dst = torch.empty(8, 8, device=gpu)
        ops.stage_inputs([(dst, src)], pos, 4)
        assert torch.equal(dst.cpu(), src.float().cpu().expand(8, 8)) and pos.item() == 4
    with pytest.raises(RuntimeError):
        ops.stage_inputs([(torch.empty(8, 8, device=gpu), torch.empty(3, 5, device=gpu))], pos, 4)
