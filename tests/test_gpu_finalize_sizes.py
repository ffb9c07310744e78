"""npu_moe_finalize_routing in bf16 at the sizes where its launch changes: the few-token form (up to 256 tokens,
64-thread workgroups over the columns) and the other, ends of a column chunk, more experts per token than are in
flight at once, dropped rows whose would-be source holds NaN, skips and bias. Bound: the fp32 sums are the
oracle's in the same order, the output one bf16 rounding, so equal bit for bit to a float32 reference summed in
slot order."""
import numpy as np
import pytest
import torch

import torchair_amd  # noqa: F401

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("t", [1, 256, 257])
@pytest.mark.parametrize("h,k", [(8, 1), (520, 2), (520, 3), (520, 4), (520, 5), (504, 8), (520, 9), (7168, 8), (520, 17)])
def test_finalize_sizes(t, h, k):
    g = torch.Generator().manual_seed(t + h + k)
    ex = torch.randn(t * k + 1, h, generator=g).to(torch.bfloat16)
    ex[-1] = float("nan")
    dst = torch.randperm(t * k, generator=g).to(torch.int32)
    drop = torch.rand(t * k, generator=g) < 0.1
    dst[drop] = -1
    scales = torch.rand(t, k, generator=g)
    skip = torch.randn(t, h, generator=g).to(torch.bfloat16)
    bias = torch.randn(5, h, generator=g).to(torch.bfloat16)
    expert = torch.randint(0, 5, (t, k), generator=g, dtype=torch.int32)
    print("case", t, h, k, flush=True)
    y = torch.ops.npu.npu_moe_finalize_routing(ex.to(DEV), skip.to(DEV), None, bias.to(DEV), scales.to(DEV), dst.to(DEV),
                                               expert.to(DEV), drop_pad_mode=2)
    e, d = ex.float().numpy(), dst.view(t, k).numpy()
    acc = skip.float().numpy().copy()
    for j in range(k):
        live = d[:, j] >= 0
        v = e[d[live, j]] + bias.float().numpy()[expert[:, j].numpy()[live]]
        acc[live] = acc[live] + scales[:, j].numpy()[live, None] * v
    assert torch.equal(y.cpu(), torch.from_numpy(acc.astype(np.float32)).to(torch.bfloat16))
