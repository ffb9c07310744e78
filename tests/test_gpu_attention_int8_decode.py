"""One-token paged decode over int8 caches with per-channel scales, against 64-bit attention on the same
integers: head dims, group sizes, both 16-bit query types, caches that start on 8 bytes only, sequences around
the 32-token step and over many ranges, scores that rise along the keys, and queries far from 1.

Bound: the query times the key scale has 22 bits, P is rounded to fp16 (2^-12 of each term) and the output to its
type. The first tests allow a query rounded once to fp16 (2^-12 of each product): |o - w| <= u |w| + (2^-11 + 2 d)
max|v|, u = 2^-8 (bf16) or 2^-11 (fp16) and d = 2^-12 scale max_j sum|q ks k_j|, the largest error of a score; the
last one takes d = 2^-20 scale max_j sum|q ks k_j|, 22 bits and sums in fp32."""
import math

import numpy as np
import pytest
import torch

import torchair_amd  # noqa: F401

pytestmark = pytest.mark.gpu
DEV = "cuda"
FIA = torch.ops.air.npu_fused_infer_attention_score


def _case(d, hq, hkv, dt, bs, lens, seed, shift=0, qstd=1.0, ramp=False, bnsd=False):
    g = torch.Generator().manual_seed(seed)
    nb = [max(1, -(-n // bs)) for n in lens]
    total = sum(nb) + 1
    perm = torch.randperm(total, generator=g).to(torch.int32)
    bt = torch.zeros(len(lens), max(nb), dtype=torch.int32)
    at = 0
    for i, n in enumerate(nb):
        bt[i, :n] = perm[at:at + n]
        at += n
    shape = (total, hkv, bs, d) if bnsd else (total, bs, hkv * d)
    caches = []
    for _ in range(2):
        flat = torch.randint(-128, 128, (math.prod(shape) + shift,), generator=g, dtype=torch.int8).to(DEV)
        caches.append(flat[shift:].view(shape))
    if ramp:  # keys that grow with the position: the reference max is raised many times
        for b, n in enumerate(lens):
            for p in range(-(-n // bs)):
                page = int(bt[b, p])
                caches[0][page] = (caches[0][page].float() * min(1.0, (p + 1) / 12)).to(torch.int8)
    q = (torch.randn(len(lens), 1, hq * d, generator=g) * qstd).to(dt).to(DEV)
    ks, vs = [(torch.rand(hkv * d, generator=g) * 0.03 + 0.005).to(DEV) for _ in range(2)]
    print("case", d, hq, hkv, dt, bs, lens, shift, flush=True)
    out, lse = FIA(q, caches[0], caches[1], actual_seq_lengths_kv=torch.tensor(lens, device=DEV), block_table=bt.to(DEV),
                   num_heads=hq, num_key_value_heads=hkv, input_layout="BSH", block_size=bs, scale=d ** -0.5,
                   key_antiquant_scale=ks, value_antiquant_scale=vs, softmax_lse_flag=True)
    k4, v4 = [(c.transpose(1, 2) if bnsd else c.view(total, bs, hkv, d)).cpu().numpy().astype(np.float64) for c in caches]
    k4, v4 = k4 * ks.double().cpu().numpy().reshape(hkv, d), v4 * vs.double().cpu().numpy().reshape(hkv, d)
    qn = q.double().cpu().numpy().reshape(len(lens), hq, d)
    got, gl = out.double().cpu().numpy().reshape(len(lens), hq, d), lse.cpu().numpy().reshape(len(lens), hq)
    u = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -11
    for b, n in enumerate(lens):
        if n == 0:
            assert (got[b] == 0).all() and np.isneginf(gl[b]).all()
            continue
        pages = bt[b, :-(-n // bs)].numpy()
        k, v = k4[pages].reshape(-1, hkv, d)[:n], v4[pages].reshape(-1, hkv, d)[:n]
        for h in range(hq):
            kh, vh = k[:, h // (hq // hkv)], v[:, h // (hq // hkv)]
            s = kh @ qn[b, h] * d ** -0.5
            err = 2.0 ** -12 * d ** -0.5 * (np.abs(kh) @ np.abs(qn[b, h])).max()
            p = np.exp(s - s.max())
            w = p @ vh / p.sum()
            assert (np.abs(got[b, h] - w) <= u * np.abs(w) + (2.0 ** -11 + 2 * err) * np.abs(vh).max()).all(), (b, h)
            assert abs(gl[b, h] - (s.max() + np.log(p.sum()))) <= err + 1e-3


@pytest.mark.parametrize("shift", [0, 8])
@pytest.mark.parametrize("d,hq,hkv,dt", [(128, 8, 2, torch.bfloat16), (64, 16, 1, torch.float16),
                                         (256, 7, 1, torch.bfloat16), (128, 4, 4, torch.float16)])
def test_int8_decode(d, hq, hkv, dt, shift):
    _case(d, hq, hkv, dt, 64, [0, 1, 31, 32, 33, 64, 200, 1100], 400 + d + hq, shift)


def test_int8_decode_long_sequences_and_head_major_pages():
    _case(128, 8, 1, torch.bfloat16, 32, [9000, 5], 410)
    _case(128, 8, 2, torch.float16, 128, [700, 129, 1], 411, bnsd=True)


@pytest.mark.parametrize("qstd", [30.0, 1e-4, 3000.0])
def test_int8_decode_query_ranges_and_rising_scores(qstd):
    """Queries whose products lie far outside fp16, and keys whose scores rise page by page."""
    _case(128, 8, 2, torch.bfloat16, 32, [500, 90], 420, qstd=qstd if qstd < 100 else 3.0, ramp=True)
    _case(64, 4, 1, torch.bfloat16, 64, [77], 421, qstd=qstd)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("mean,std,ints", [(0.0, 3.0, 32), (4.0, 0.1, 32), (4.0, 0.1, 1)])
def test_int8_decode_scores_keep_their_precision(d, dt, mean, std, ints):
    """Large scores, queries of one sign and keys of few steps, where a rounded query or sums far above the scores
    would show: the lse within 2^-11 (the row sum takes the rounded P) and the scores' own 2^-20."""
    g = torch.Generator(device=DEV).manual_seed(430 + d)
    b, n, bs, hq, hkv = 4, 700, 64, 8, 2
    nb = -(-n // bs)
    bt = torch.arange(b * nb, device=DEV, dtype=torch.int32).view(b, nb)
    q = (torch.randn(b, 1, hq * d, generator=g, device=DEV) * std + mean).to(dt)
    k, v = [(torch.randn(b * nb, bs, hkv * d, generator=g, device=DEV) * ints).round().clamp(-127, 127).to(torch.int8)
            for _ in range(2)]
    ks, vs = [(torch.rand(hkv * d, generator=g, device=DEV) * 0.03 + 0.01) * 32 / ints for _ in range(2)]
    print("case", d, dt, mean, std, ints, flush=True)
    out, lse = FIA(q, k, v, actual_seq_lengths_kv=torch.tensor([n] * b, device=DEV), block_table=bt, num_heads=hq,
                   num_key_value_heads=hkv, input_layout="BSH", block_size=bs, scale=d ** -0.5, key_antiquant_scale=ks,
                   value_antiquant_scale=vs, softmax_lse_flag=True)
    u = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -11
    k, v = [(x.double() * y.double()).cpu().numpy().reshape(b, nb * bs, hkv, d)[:, :n] for x, y in ((k, ks), (v, vs))]
    q, out, lse = q.double().cpu().numpy().reshape(b, hq, d), out.double().cpu().numpy().reshape(b, hq, d), lse.cpu().numpy()
    for i in range(b):
        for h in range(hq):
            kh, vh = k[i, :, h // (hq // hkv)], v[i, :, h // (hq // hkv)]
            s = kh @ q[i, h] * d ** -0.5
            err = 2.0 ** -20 * d ** -0.5 * (np.abs(kh) @ np.abs(q[i, h])).max()
            p = np.exp(s - s.max())
            w = p @ vh / p.sum()
            assert (np.abs(out[i, h] - w) <= u * np.abs(w) + (2.0 ** -11 + 2 * err) * np.abs(vh).max()).all(), (i, h)
            assert abs(lse.reshape(b, hq)[i, h] - (s.max() + np.log(p.sum()))) <= 2.0 ** -11 + err
