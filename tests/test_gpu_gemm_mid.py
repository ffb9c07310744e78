"""Dense W8A8 GEMMs of 128 to 2048 rows, where the tile shape and the K split change with the size: exact int32
accumulators against an int64 product, and the bf16 epilogue bit for bit against the documented order of
operations, for [K, N] and [N, K] weights."""
import pytest
import torch

import torchair_amd  # noqa: F401
from torchair_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("m", [129, 255, 256, 257, 384, 1023, 2049])
@pytest.mark.parametrize("k,n", [(64, 256), (1536, 512), (4160, 272), (5632, 2048), (1024, 4112)])
@pytest.mark.parametrize("nk", [False, True])
def test_mid_rows(m, k, n, nk):
    g = torch.Generator(device=DEV).manual_seed(m + k + n)
    x = torch.randint(-128, 128, (m, k), generator=g, device=DEV, dtype=torch.int8)
    w = torch.randint(-128, 128, (k, n), generator=g, device=DEV, dtype=torch.int8)
    wt = w.t().contiguous().t() if nk else w
    want = (x.double() @ w.double())  # exact: below 2^53
    print("case", m, k, n, nk, flush=True)
    acc = torch.ops.npu.npu_quant_matmul(x, wt, torch.ones(1, device=DEV), output_dtype=torch.int32)
    assert torch.equal(acc.double(), want)
    scale = torch.rand(n, generator=g, device=DEV) * 1e-3
    pt = torch.rand(m, generator=g, device=DEV)
    bias = torch.randn(n, generator=g, device=DEV)
    y = torch.ops.npu.npu_quant_matmul(x, wt, scale, pertoken_scale=pt, bias=bias, output_dtype=torch.bfloat16)
    ref = ((acc.float() * scale) * pt[:, None] + bias).to(torch.bfloat16)
    assert torch.equal(y, ref)


def test_no_workspace():
    """From 256 rows on, a direct call without a workspace stays accepted and gives the same accumulators."""
    m, k, n = 300, 4096, 512
    assert _lib.query("tai_quant_matmul_workspace_size", m, k, n, _lib.DT_INT32) > 0  # a split is wanted
    g = torch.Generator(device=DEV).manual_seed(1)
    x = torch.randint(-128, 128, (m, k), generator=g, device=DEV, dtype=torch.int8)
    w = torch.randint(-128, 128, (k, n), generator=g, device=DEV, dtype=torch.int8)
    out = torch.empty(m, n, device=DEV, dtype=torch.int32)
    _lib.call("tai_quant_matmul", x.data_ptr(), w.data_ptr(), m, k, n, _lib.LAYOUT_KN, None, 0, None, 0, None, None,
              _lib.DT_NONE, _lib.DT_INT32, out.data_ptr(), None, 0, torch.cuda.current_stream().cuda_stream)
    assert torch.equal(out.double(), x.double() @ w.double())


@pytest.mark.parametrize("m", [256, 300])
@pytest.mark.parametrize("k", [16, 32, 48])
@pytest.mark.parametrize("nk", [False, True])
def test_short_k(m, k, nk):
    """K below one 64-byte stage, which no split plan takes: the 128-row tiles, with every output type."""
    n = 512
    g = torch.Generator(device=DEV).manual_seed(m + k)
    x = torch.randint(-128, 128, (m, k), generator=g, device=DEV, dtype=torch.int8)
    w = torch.randint(-128, 128, (k, n), generator=g, device=DEV, dtype=torch.int8)
    wt = w.t().contiguous().t() if nk else w
    want = x.double() @ w.double()
    print("case", m, k, nk, flush=True)
    acc = torch.ops.npu.npu_quant_matmul(x, wt, torch.ones(1, device=DEV), output_dtype=torch.int32)
    assert torch.equal(acc.double(), want)
    scale = torch.rand(n, generator=g, device=DEV) * 1e-3
    y = torch.ops.npu.npu_quant_matmul(x, wt, scale, output_dtype=torch.bfloat16)
    assert torch.equal(y, (acc.float() * scale).to(torch.bfloat16))
    y8 = torch.ops.npu.npu_quant_matmul(x, wt, scale, output_dtype=torch.int8)
    assert torch.equal(y8, (acc.float() * scale).round().clamp(-128, 127).to(torch.int8))
