"""tai_fia_tiled against tai_fia_general: every call the tiled kernels take is also the general kernel's, with
the same arguments, so the two are run on the same inputs. Both keep scores, probabilities, sums and O in fp32
precision and round the output once to 16 bits, so they differ by at most one rounding step of the output plus
fp32 sums in another order: |a - b| <= 2^-7 |b| (bf16; 2^-10 fp16) + 2^-14 max|v|, and lse by 1e-4 of max(1, |lse|).
The last tests compare both kernels with 64-bit attention that shares none of their code."""
import math

import numpy as np
import pytest
import torch

import torchair_amd  # noqa: F401
from torchair_amd import _fia, _lib

pytestmark = pytest.mark.gpu
DEV = "cuda"
FIA = torch.ops.air.npu_fused_infer_attention_score
FIA2 = torch.ops.air.npu_fused_infer_attention_score_v2


def _both(monkeypatch, call):
    """(tiled result, general result); fails if the tiled kernels do not take the call."""
    taken = []
    real = _lib.query

    def spy(name, *args):
        n = real(name, *args)
        if name == "tai_fia_tiled_workspace_size":
            taken.append(n)
        return n

    monkeypatch.setattr(_fia._lib, "query", spy)
    tiled = call()
    assert taken and taken[-1] > 0, "the call did not reach the tiled kernels"
    monkeypatch.setattr(_fia._lib, "query", lambda name, *a: 0 if name == "tai_fia_tiled_workspace_size" else real(name, *a))
    general = call()
    monkeypatch.setattr(_fia._lib, "query", real)
    return tiled, general


def _assert_same(tiled, general, vmax):
    (o, l), (wo, wl) = tiled, general
    assert o.dtype == wo.dtype and o.shape == wo.shape
    o, wo = o.float().cpu().numpy(), wo.float().cpu().numpy()
    assert np.array_equal(np.isfinite(o), np.isfinite(wo))
    fine = np.isfinite(wo)
    step = 2.0 ** -7 if tiled[0].dtype == torch.bfloat16 else 2.0 ** -10
    assert (np.abs(o[fine] - wo[fine]) <= step * np.abs(wo[fine]) + 2.0 ** -14 * vmax).all()
    l, wl = l.cpu().numpy(), wl.cpu().numpy()
    assert l.shape == wl.shape and np.array_equal(np.isfinite(l), np.isfinite(wl))
    fine = np.isfinite(wl)
    assert (np.abs(l[fine] - wl[fine]) <= 1e-4 * np.maximum(1, np.abs(wl[fine]))).all()


def _table(lens, bs, g, spare=2):
    nb = [max(1, -(-n // bs)) for n in lens]
    perm = torch.randperm(sum(nb) + spare, generator=g).to(torch.int32)
    bt = torch.zeros(len(lens), max(nb), dtype=torch.int32)
    at = 0
    for i, n in enumerate(nb):
        bt[i, :n] = perm[at:at + n]
        at += n
    return bt, sum(nb) + spare


# ------------------------------------------------------------------------------------------------ MLA, bf16 latent
def _mla(lens, hq, sq, bs, seed, layout="BSND", std=1.0):
    g = torch.Generator().manual_seed(seed)
    bt, n = _table(lens, bs, g)
    shape = (len(lens), sq, hq) if layout == "BSND" else (len(lens), hq, sq)
    qn = (torch.randn(*shape, 512, generator=g) * std).to(torch.bfloat16)
    qr = torch.randn(*shape, 64, generator=g).to(torch.bfloat16)
    c = (torch.randn(n, bs, 1, 512, generator=g) * 0.7).to(torch.bfloat16)
    kr = torch.randn(n, bs, 1, 64, generator=g).to(torch.bfloat16)
    return [t.to(DEV) for t in (qn, qr, c, kr, bt)]


def _mla_call(t, lens, hq, bs, layout="BSND", **kw):
    qn, qr, c, kr, bt = t
    return lambda: FIA(qn, c, c, query_rope=qr, key_rope=kr, block_table=bt, num_heads=hq, num_key_value_heads=1,
                       actual_seq_lengths_kv=torch.tensor(lens, device=DEV), input_layout=layout, block_size=bs,
                       scale=192 ** -0.5, softmax_lse_flag=True, **kw)


@pytest.mark.parametrize("lens,hq,sq,bs", [
    ([1], 16, 1, 32),                                # one step, one range
    ([31, 32, 33, 0, 64, 65], 128, 1, 64),           # edges of a step, an empty sequence
    ([300, 1, 129], 40, 1, 128),                     # heads that fill no head block
    ([5000], 128, 1, 128),                           # one sequence over many ranges
    ([2100, 70, 2049], 136, 2, 32),                  # two head groups, two query tokens, more than 64 pages
    ([4, 1, 0, 700], 64, 5, 64),                     # fewer keys than query tokens
])
def test_mla_rows(monkeypatch, lens, hq, sq, bs):
    t = _mla(lens, hq, sq, bs, 200 + hq + sq)
    for kw in ([{}, {"sparse_mode": 3}, {"sparse_mode": 2}] if sq > 1 else [{}]):
        tiled, general = _both(monkeypatch, _mla_call(t, lens, hq, bs, **kw))
        _assert_same(tiled, general, 4.0)


def test_mla_rows_many_short(monkeypatch):
    """More rows than a workgroup scans itself, most of them whole inside one range."""
    lens = [(7 * i) % 90 for i in range(150)]
    t = _mla(lens, 32, 3, 32, 211, layout="BNSD")
    _assert_same(*_both(monkeypatch, _mla_call(t, lens, 32, 32, layout="BNSD", sparse_mode=3,
                                               actual_seq_lengths=torch.tensor([i % 4 for i in range(150)], device=DEV))), 4.0)


def test_mla_rows_packed_and_sink(monkeypatch):
    g = torch.Generator().manual_seed(212)
    lq, lk, hq, bs = [1, 4, 0, 2], [300, 260, 5, 33], 24, 64
    bt, n = _table(lk, bs, g)
    qn = torch.randn(sum(lq) + 2, hq, 512, generator=g).to(torch.bfloat16).to(DEV)
    qr = torch.randn(sum(lq) + 2, hq, 64, generator=g).to(torch.bfloat16).to(DEV)
    c = torch.randn(n, bs, 1, 512, generator=g).to(torch.bfloat16).to(DEV)
    kr = torch.randn(n, bs, 1, 64, generator=g).to(torch.bfloat16).to(DEV)
    sink = torch.randn(hq, generator=g)
    sink[3] = -math.inf
    _assert_same(*_both(monkeypatch, lambda: FIA2(
        qn, c, c, query_rope=qr, key_rope=kr, block_table=bt.to(DEV), num_query_heads=hq, num_key_value_heads=1,
        actual_seq_qlen=torch.tensor(np.cumsum(lq), device=DEV), actual_seq_kvlen=torch.tensor(lk, device=DEV),
        input_layout="TND", block_size=bs, softmax_scale=192 ** -0.5, return_softmax_lse=True, sparse_mode=3,
        learnable_sink=sink.to(torch.bfloat16).to(DEV))), 4.0)


def test_mla_rows_rising_logits_and_unread_cache(monkeypatch):
    """Scores that rise far above the first step's (the reference max is raised again and again), and NaN and
    infinities in the cache slots that no query sees."""
    lens, hq, bs = [260, 100], 16, 64
    qn, qr, c, kr, bt = _mla(lens, hq, 1, bs, 213, std=6.0)
    for b, n in enumerate(lens):
        for p in range(-(-n // bs)):
            page = int(bt[b, p])
            ramp = torch.arange(p * bs, (p + 1) * bs, device=DEV).float().view(bs, 1, 1) / 16
            c[page] = (c[page].float() * ramp).to(torch.bfloat16)
            if (p + 1) * bs > n:
                c[page, n - p * bs:] = math.nan
                kr[page, n - p * bs:] = math.inf
    _assert_same(*_both(monkeypatch, _mla_call((qn, qr, c, kr, bt), lens, hq, bs)), 60.0)


# ------------------------------------------------------------------------------------------------ GQA/MHA blocks
def _kv(n, bs, hkv, d, dt, g, bnsd=False):
    shape = (n, hkv, bs, d) if bnsd else (n, bs, hkv * d)
    return [torch.randn(*shape, generator=g).to(dt).to(DEV) for _ in range(2)]


def _packed(monkeypatch, lq, lk, hq, hkv, d, bs, seed, dt=torch.bfloat16, layout="TND", pad=0, bnsd=False, edit=None,
            scale=None, v2=False, **kw):
    g = torch.Generator().manual_seed(seed)
    bt, n = _table(lk, bs, g)
    k, v = _kv(n, bs, hkv, d, dt, g, bnsd)
    q = torch.randn(sum(lq) + pad, hq, d, generator=g).to(dt).to(DEV)
    if edit:
        edit(q, k, v, bt)
    ends = torch.tensor(np.cumsum(lq), device=DEV)
    lens = torch.tensor(lk, device=DEV)
    scale = d ** -0.5 if scale is None else scale
    if v2:
        return _both(monkeypatch, lambda: FIA2(q, k, v, actual_seq_qlen=ends, actual_seq_kvlen=lens, block_table=bt.to(DEV),
                                               num_query_heads=hq, num_key_value_heads=hkv, input_layout=layout,
                                               block_size=bs, softmax_scale=scale, return_softmax_lse=True, **kw))
    return _both(monkeypatch, lambda: FIA(q, k, v, actual_seq_lengths=ends, actual_seq_lengths_kv=lens,
                                          block_table=bt.to(DEV), num_heads=hq, num_key_value_heads=hkv,
                                          input_layout=layout, block_size=bs, scale=scale, softmax_lse_flag=True, **kw))


@pytest.mark.parametrize("lq,lk,hq,hkv,d,bs", [
    ([1], [1], 4, 4, 128, 32),                                      # one column, one token
    ([1] * 9, [63, 64, 65, 1, 0, 700, 128, 31, 2000], 32, 8, 128, 128),
    ([64, 65, 0, 63, 1], [64, 300, 40, 63, 1500], 32, 8, 128, 64),  # edges of a block of columns
    ([37, 5], [37, 1000], 28, 4, 128, 96),                          # 7 heads a group, pages of 96
    ([130, 3], [130, 3000], 8, 8, 64, 32),                          # one head a group, a tile over two pages
    ([20, 33, 1], [900, 33, 4000], 64, 2, 64, 128),                 # 32 heads a group
    ([300, 1], [9, 1], 16, 2, 128, 64),                             # rows that see nothing
    ([2, 0] * 35, [2 + 5 * i for i in range(70)], 8, 2, 64, 32),    # short sequences, every other one empty
    ([512], [512], 16, 4, 128, 128),                                # the most rows that the kernel plans by itself,
    ([513], [700], 16, 4, 128, 128),                                # and one more
    ([1, 0, 2, 1] * 128, [(7 * i) % 90 for i in range(512)], 4, 2, 64, 32),        # the most sequences that it does,
    ([1, 0, 2, 1] * 128 + [1], [(7 * i) % 90 for i in range(513)], 4, 2, 64, 32),  # and one more
    ([300] + [1] * 15 + [280, 0, 1], [300] + [40] * 15 + [500, 9, 77], 16, 2, 64, 32),  # long ones in one planning wave
])
@pytest.mark.parametrize("mode", [{"sparse_mode": 3}, {}, {"sparse_mode": 4, "pre_tokens": 70, "next_tokens": 9}])
def test_packed_paged(monkeypatch, lq, lk, hq, hkv, d, bs, mode):
    _assert_same(*_packed(monkeypatch, lq, lk, hq, hkv, d, bs, 300 + hq, **mode), 4.5)


@pytest.mark.parametrize("layout", ["TND", "TND_NTD"])
def test_packed_layouts_fp16_padding(monkeypatch, layout):
    """fp16, rows past the last end (zeros, lse -inf), head-major pages."""
    _assert_same(*_packed(monkeypatch, [5, 70, 1], [200, 70, 513], 16, 4, 128, 64, 310, dt=torch.float16, layout=layout,
                          pad=67, bnsd=True, sparse_mode=3), 4.5)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("scale", [0.3, -0.2, 0.0])
def test_packed_scales_and_rising_logits(monkeypatch, dt, scale):
    """Scores that rise along the keys (raised reference maxima), a negative and a zero scale."""
    def rise(q, k, v, bt):
        for b, n in enumerate([600, 900]):
            for p in range(-(-n // 64)):
                k[int(bt[b, p])] *= 0.2 + p
    _assert_same(*_packed(monkeypatch, [40, 1], [600, 900], 8, 2, 64, 64, 320, dt=dt, scale=scale, edit=rise,
                          sparse_mode=3), 4.5)


def test_packed_nan_scale(monkeypatch):
    """A scale of NaN gives NaN wherever a row sees a key, as in the general kernel."""
    tiled, general = _packed(monkeypatch, [5, 0, 1], [70, 9, 300], 8, 2, 64, 64, 321, scale=math.nan, sparse_mode=3)
    assert torch.isnan(general[0]).all() and torch.isnan(tiled[0]).all()
    assert torch.equal(tiled[1], general[1])


def test_packed_sink(monkeypatch):
    sink = torch.linspace(-3, 6, 16)
    sink[5] = -math.inf
    _assert_same(*_packed(monkeypatch, [40, 0, 1, 7], [600, 3, 900, 2], 16, 4, 128, 64, 330, v2=True, sparse_mode=3,
                          learnable_sink=sink.to(torch.bfloat16).to(DEV)), 4.5)


def test_packed_values_that_are_not_finite(monkeypatch):
    """NaN and infinities in slots that no query sees, and an infinite value that only later rows see: the rows
    before it stay finite."""
    def spoil(q, k, v, bt):
        for b, n in enumerate([600, 100, 2000]):
            page, slot = int(bt[b, n // 64]), n % 64
            if slot:
                k[page, slot:] = math.nan
                v[page, slot:] = math.inf
        v[int(bt[0, 590 // 64]), 590 % 64, 3] = math.inf   # seen by the last 10 of the 40 rows
        v[int(bt[2, 1990 // 64]), 1990 % 64, 70] = math.nan  # the same in an item cut over several ranges
        k[int(bt[2, 3]), 5, 9] = -math.inf  # scores of +-inf (kv head 0) ...
        k[int(bt[2, 4]), 5, 9] = math.inf   # ... and so rows of NaN
    tiled, general = _packed(monkeypatch, [40, 20, 50], [600, 100, 2000], 8, 2, 128, 64, 340, sparse_mode=3, edit=spoil)
    assert np.isfinite(general[0].float().cpu().numpy()[:20]).all()
    _assert_same(tiled, general, 4.5)


@pytest.mark.parametrize("d,dt", [(128, torch.bfloat16), (64, torch.float16)])
def test_packed_dense_keys(monkeypatch, d, dt):
    """Keys packed like the queries (no pages), top-left causal; and a batched prefill with a sink."""
    g = torch.Generator().manual_seed(350)
    lq, lk, hq, hkv = [33, 1, 70, 0], [33, 5, 290, 4], 8, 2
    q = torch.randn(sum(lq) + 3, hq, d, generator=g).to(dt).to(DEV)
    k, v = [torch.randn(sum(lk) + 2, hkv, d, generator=g).to(dt).to(DEV) for _ in range(2)]
    for mode, layout in ((2, "TND"), (3, "TND"), (3, "NTD"), (3, "NTD_TND")):
        args = [t.transpose(0, 1).contiguous() if layout.startswith("NTD") else t for t in (q, k, v)]
        _assert_same(*_both(monkeypatch, lambda: FIA(
            *args, actual_seq_lengths=torch.tensor(np.cumsum(lq), device=DEV),
            actual_seq_lengths_kv=torch.tensor(np.cumsum(lk), device=DEV), num_heads=hq, num_key_value_heads=hkv,
            input_layout=layout, scale=d ** -0.5, sparse_mode=mode, softmax_lse_flag=True)), 4.5)
    sink = torch.randn(hq, generator=g).to(torch.bfloat16).to(DEV)
    for layout in ("BSND", "BNSD"):
        sh = (lambda s, n: (3, s, n, d)) if layout == "BSND" else (lambda s, n: (3, n, s, d))
        q4 = torch.randn(*sh(75, hq), generator=g).to(dt).to(DEV)
        k4, v4 = [torch.randn(*sh(200, hkv), generator=g).to(dt).to(DEV) for _ in range(2)]
        _assert_same(*_both(monkeypatch, lambda: FIA2(
            q4, k4, v4, actual_seq_qlen=torch.tensor([75, 10, 0], device=DEV),
            actual_seq_kvlen=torch.tensor([200, 10, 7], device=DEV), num_query_heads=hq, num_key_value_heads=hkv,
            input_layout=layout, softmax_scale=d ** -0.5, return_softmax_lse=True, sparse_mode=3,
            learnable_sink=sink)), 4.5)


def test_packed_rows_off_16_bytes_take_the_general_kernel(monkeypatch):
    g = torch.Generator().manual_seed(360)
    hq, hkv, d, bs, lq, lk = 4, 2, 128, 64, [5, 9], [70, 9]
    bt, n = _table(lk, bs, g)
    k, v = _kv(n, bs, hkv, d, torch.bfloat16, g)
    wide = torch.randn(sum(lq), hq, d + 1, generator=g).to(torch.bfloat16).to(DEV)
    call = lambda q: FIA(q, k, v, actual_seq_lengths=torch.tensor(np.cumsum(lq), device=DEV),  # noqa: E731
                         actual_seq_lengths_kv=torch.tensor(lk, device=DEV), block_table=bt.to(DEV), num_heads=hq,
                         num_key_value_heads=hkv, input_layout="TND", block_size=bs, scale=d ** -0.5, sparse_mode=3,
                         softmax_lse_flag=True)
    sizes = []
    real = _lib.query
    monkeypatch.setattr(_fia._lib, "query", lambda name, *a: sizes.append(real(name, *a)) or sizes[-1])
    off = call(wide[..., 1:])
    assert sizes[-1] == 0
    _assert_same(call(wide[..., 1:].contiguous()), off, 4.5)
    assert sizes[-1] > 0


@pytest.mark.parametrize("bs", [32, 96])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
def test_packed_band_does_not_read_released_pages(bs, dt):
    """A sliding window whose lower edge lies inside a 64-token tile but past that tile's first page: pages below the
    band may have left the block table. They name a page of NaN and infinities here, whose values would send the
    block to the plain fp32 path; the result equals, bit for bit, that with the pages still in the table."""
    g = torch.Generator().manual_seed(370 + bs)
    hq, hkv, d, pre = 8, 2, 128, 130
    lq, lk = [1, 5, 70], [231, 1000, 560]  # lower edges at 100, 865 and 360
    bt, n = _table(lk, bs, g)
    k, v = _kv(n, bs, hkv, d, dt, g)
    spare = (set(range(n)) - {int(p) for row, m in zip(bt, lk) for p in row[:-(-m // bs)]}).pop()
    k[spare], v[spare] = math.nan, math.inf
    q = torch.randn(sum(lq), hq, d, generator=g).to(dt).to(DEV)
    gone = bt.clone()
    for b, (nq, nk) in enumerate(zip(lq, lk)):
        gone[b, :(nk - nq - pre) // bs] = spare
    assert (gone != bt).any(1).all()
    print("case", bs, dt, flush=True)
    call = lambda t: FIA(q, k, v, actual_seq_lengths=torch.tensor(np.cumsum(lq), device=DEV),  # noqa: E731
                         actual_seq_lengths_kv=torch.tensor(lk, device=DEV), block_table=t.to(DEV), num_heads=hq,
                         num_key_value_heads=hkv, input_layout="TND", block_size=bs, scale=d ** -0.5, sparse_mode=4,
                         pre_tokens=pre, next_tokens=0, softmax_lse_flag=True)
    want, got = call(bt), call(gone)
    assert np.isfinite(want[0].float().cpu().numpy()).all()
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


def _guarded(monkeypatch, call):
    """(call's result, workspace bytes) with 1 MB of a pattern behind the workspace, which must stay as it was."""
    real, seen = _lib.call, []

    def spy(name, *args):
        if name != "tai_fia_tiled":
            return real(name, *args)
        a, _, n, stream = args
        buf = torch.full((n + (1 << 20),), 0x5A, dtype=torch.uint8, device=DEV)
        real(name, a, buf.data_ptr(), n, stream)
        assert bool((buf[n:] == 0x5A).all()), "written past the workspace"
        seen.append(n)

    monkeypatch.setattr(_fia._lib, "call", spy)
    out = call()
    monkeypatch.setattr(_fia._lib, "call", real)
    assert len(seen) == 1
    return out, seen[0]


@pytest.mark.parametrize("lq,lk,hq,hkv,d,bs,most", [
    ([1], [1], 4, 4, 64, 32, 1 << 18),
    ([1] * 4, [128, 7, 64, 128], 32, 8, 128, 128, 1 << 21),
    ([3, 0, 9], [500, 4, 9], 16, 2, 128, 64, 1 << 24),
    ([30] * 3, [200, 30, 77], 8, 8, 64, 32, 1 << 23),                  # one wave of columns a block
    ([40] * 3, [200, 40, 77], 16, 4, 128, 32, 1 << 25),                # five
    ([200, 1, 60], [3000, 2000, 60], 32, 8, 128, 128, 66 << 20),        # 256 ranges of 256 columns
])
def test_packed_workspace_follows_the_call(monkeypatch, lq, lk, hq, hkv, d, bs, most):
    """Small calls take a small workspace and stay inside it, and equal the general kernel."""
    g = torch.Generator().manual_seed(380 + hq + len(lq))
    bt, n = _table(lk, bs, g)
    k, v = _kv(n, bs, hkv, d, torch.bfloat16, g)
    q = torch.randn(sum(lq) + 2, hq, d, generator=g).to(torch.bfloat16).to(DEV)
    print("case", lq, lk, hq, hkv, d, bs, flush=True)
    call = lambda: FIA(q, k, v, actual_seq_lengths=torch.tensor(np.cumsum(lq), device=DEV),  # noqa: E731
                       actual_seq_lengths_kv=torch.tensor(lk, device=DEV), block_table=bt.to(DEV), num_heads=hq,
                       num_key_value_heads=hkv, input_layout="TND", block_size=bs, scale=d ** -0.5, sparse_mode=3,
                       softmax_lse_flag=True)
    got, size = _guarded(monkeypatch, call)
    assert size <= most
    _assert_same(got, _both(monkeypatch, call)[1], 4.5)


@pytest.mark.parametrize("lens,hq,sq,bs,most", [
    ([1], 16, 1, 32, 1 << 20),
    ([128], 128, 1, 128, 6 << 20),
    ([64, 0, 3], 40, 2, 32, 6 << 20),
    ([100, 31], 136, 1, 32, 23 << 20),
    ([4000] * 3, 128, 1, 128, 129 << 20),  # 256 ranges of 128 heads
])
def test_mla_rows_workspace_follows_the_call(monkeypatch, lens, hq, sq, bs, most):
    call = _mla_call(_mla(lens, hq, sq, bs, 390 + hq), lens, hq, bs)
    print("case", lens, hq, sq, bs, flush=True)
    got, size = _guarded(monkeypatch, call)
    assert size <= most
    _assert_same(got, _both(monkeypatch, call)[1], 4.0)


# ------------------------------------------------------------------------------------------------ against 64 bits
def _attend64(q, k, v, scale):
    """Bottom-right causal attention of q [lq, hq, dk] over k [lk, hkv, dk], v [lk, hkv, dv]: (out, lse)."""
    lq, lk, rep = q.shape[0], k.shape[0], q.shape[1] // k.shape[1]
    s = np.einsum("ihd,jhd->hij", q, np.repeat(k, rep, 1)) * scale
    s = np.where(np.arange(lk)[None] <= np.arange(lq)[:, None] + lk - lq, s, -np.inf)
    m = s.max(-1, keepdims=True)
    p = np.exp(s - m)
    l = p.sum(-1, keepdims=True)
    return np.einsum("hij,jhd->ihd", p / l, np.repeat(v, rep, 1)), (m + np.log(l))[..., 0].T


def _check64(out, lse, want, wlse, vmax, dt):
    """One rounding of the output (8 significant bits round by up to 2^-8 of the value, 11 by 2^-11), P as a 16-bit
    pair (2^-17 of a term) and fp32 scores and sums, 2^-15 of the largest value in all."""
    u = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -11
    far = np.abs(out.double().cpu().numpy() - want) - 1.01 * u * np.abs(want)
    assert far.max() <= 2.0 ** -15 * vmax
    assert np.abs((lse.double().cpu().numpy() - wlse) / np.maximum(1, np.abs(wlse))).max() <= 1e-5


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,d,bs", [(8, 2, 128, 64), (7, 1, 128, 96), (4, 4, 64, 32)])
def test_packed_against_64_bits(monkeypatch, hq, hkv, d, bs, dt):
    g = torch.Generator().manual_seed(400 + hq)
    lq, lk = [1, 70, 5, 1, 33], [700, 70, 260, 1, 900]
    bt, n = _table(lk, bs, g)
    k, v = _kv(n, bs, hkv, d, dt, g)
    q = (torch.randn(sum(lq), hq, d, generator=g) * 2).to(dt).to(DEV)
    both = _both(monkeypatch, lambda: FIA(
        q, k, v, actual_seq_lengths=torch.tensor(np.cumsum(lq), device=DEV),
        actual_seq_lengths_kv=torch.tensor(lk, device=DEV), block_table=bt.to(DEV), num_heads=hq,
        num_key_value_heads=hkv, input_layout="TND", block_size=bs, scale=d ** -0.5, sparse_mode=3, softmax_lse_flag=True))
    q, k, v = [x.double().cpu().numpy() for x in (q, k, v)]
    at = 0
    for i, (a, b) in enumerate(zip(lq, lk)):
        pages = bt[i, :-(-b // bs)].numpy()
        kk, vv = [x[pages].reshape(-1, hkv, d)[:b] for x in (k, v)]
        want, wlse = _attend64(q[at:at + a], kk, vv, d ** -0.5)
        for out, lse in both:
            _check64(out[at:at + a], lse[at:at + a].reshape(a, hq), want, wlse, np.abs(vv).max(), dt)
        at += a


@pytest.mark.parametrize("hq,sq", [(16, 1), (40, 3), (130, 1)])
def test_mla_rows_against_64_bits(monkeypatch, hq, sq):
    lens, bs = [sq, 33, 260, 700], 32
    t = _mla(lens, hq, sq, bs, 410 + hq)
    both = _both(monkeypatch, _mla_call(t, lens, hq, bs, sparse_mode=3))
    qn, qr, c, kr, bt = [x.double().cpu().numpy() for x in t]
    for i, n in enumerate(lens):
        pages = bt[i, :-(-n // bs)].astype(int)
        cc, rr = c[pages].reshape(-1, 1, 512)[:n], kr[pages].reshape(-1, 1, 64)[:n]
        want, wlse = _attend64(np.concatenate([qn[i], qr[i]], -1), np.concatenate([cc, rr], -1), cc, 192 ** -0.5)
        for out, lse in both:
            _check64(out[i], lse[i].reshape(hq, sq).T, want, wlse, np.abs(cc).max(), torch.bfloat16)
