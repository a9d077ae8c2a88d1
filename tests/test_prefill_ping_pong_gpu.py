"""The ping-pong prefill kernel's own cases, and the rule that chooses it, against
fp32 torch attention over the cache (INT8: through fp16, as the kernel contract
has it).  test_prefill_gpu.py runs the oracle's cases over every kernel."""
import numpy as np
import pytest

import redline_amd as ra
from tests._util import assert_close_f16, say
from tests.test_prefill_gpu import dev, run_prefill

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_cuda():
    import torch
    assert torch.cuda.is_available()
    import redline_amd.kernels  # noqa: F401
    return torch


def check_segments(torch, segs, D, kv, bs, hq, hkv, path):
    """Prefill of segs, (start, new tokens) each, under RLK_TUNE_PREFILL_DMA = path;
    every output row against fp32 attention."""
    from redline_amd import kernels as K
    from redline_amd._lib import tune_knob
    rng = np.random.default_rng(D + bs + hq)
    g = torch.Generator(device="cuda").manual_seed(D + bs + hq)
    need = [(s + n + bs - 1) // bs for s, n in segs]
    S, T, G = len(segs), sum(n for _, n in segs), hq // hkv
    cache = K.KVCache(1, sum(need) + 1, hkv, D, bs, K.KVDType.kFP16 if kv == "fp16" else K.KVDType.kINT8,
                      scale_dtype=K.SCALE_F16 if kv == "int8_f16scale" else K.SCALE_F32)
    for i, t in enumerate(x for x in cache.tensors(0) if x is not None):
        if t.dtype == torch.int8:
            t.copy_(torch.randint(-127, 128, t.shape, generator=g, device="cuda", dtype=torch.int8))
        elif i < 2:
            t.normal_(generator=g)
        else:
            t.uniform_(0.008, 0.018, generator=g)
    pool = rng.permutation(np.arange(1, sum(need) + 1, dtype=np.int32))
    bb = ra.BatchBuilder(T, S, S, max(need), bs, 1)
    tables, at = [], 0
    for (s, n), k in zip(segs, need):
        tables.append(pool[at:at + k])
        bb.add(np.zeros(n, np.int32), s, n, None, pool[at:at + k])
        at += k
    meta, shape, lay = bb.write()
    d_meta = dev(torch, meta)
    stride = (hq + 2 * hkv) * D
    q = (1.5 * torch.randn((T, stride), generator=g, device="cuda")).half()
    with tune_knob("RLK_TUNE_PREFILL_DMA", path):
        got = run_prefill(torch, K, q, stride, hq, D ** -0.5, cache.layer(0), d_meta[lay["block_tables"]:],
                          max(need), d_meta[lay["positions"]:], d_meta, lay, shape, T, D,
                          scale16=kv == "int8_f16scale")
    k, v, ks, vs = cache.tensors(0)
    at = 0
    for (s, n), t in zip(segs, tables):
        idx = torch.from_numpy(t.astype(np.int64)).cuda()
        rows = lambda x, sc: (x[idx].float() if sc is None else  # noqa: E731
                              (x[idx].float() * sc[idx].float()[..., None]).half().float()
                              ).transpose(1, 2).reshape(-1, hkv, D)[:s + n]
        kk, vv = rows(k, ks), rows(v, vs)
        mask = torch.arange(s + n, device="cuda")[None] > s + torch.arange(n, device="cuda")[:, None]
        for h in range(hq):
            sc = (q[at:at + n, h * D:(h + 1) * D].float() @ kk[:, h // G].t().contiguous()) * D ** -0.5
            want = torch.softmax(sc.masked_fill(mask, float("-inf")), -1) @ vv[:, h // G].contiguous()
            assert_close_f16(got[at:at + n, h * D:(h + 1) * D], want.cpu().numpy(), what=f"segment {s}+{n} head {h}")
        at += n


@pytest.mark.parametrize("D,kv", [(64, "fp16"), (128, "fp16"), (64, "int8"), (128, "int8"),
                                  (64, "int8_f16scale"), (128, "int8_f16scale")])
@pytest.mark.parametrize("bs,hq,hkv", [(8, 7, 1), (16, 8, 8), (16, 28, 4), (32, 24, 3), (128, 16, 2)])
def test_prefill_attention_ping_pong(torch_cuda, D, kv, bs, hq, hkv):
    """The ping-pong kernel, forced at small grids: (token, head) rows that fill
    workgroups only in part and straddle them, one tile of keys and many, tile
    ends on and off 64 keys, blocks smaller and larger than a tile, kv heads that
    do and do not divide the XCDs; against fp32 torch attention over the cache
    (INT8: through fp16, as the kernel contract has it).  Written output rows only."""
    say(f"prefill ping-pong D={D} kv={kv} bs={bs} hq={hq} hkv={hkv}")
    segs = [(0, 2), (63, 2), (0, 64), (64, 65), (200, 300), (0, 33), (447, 65), (5, 130)]
    check_segments(torch_cuda, segs, D, kv, bs, hq, hkv, 2)


@pytest.mark.parametrize("kv", ["fp16", "int8"])
@pytest.mark.parametrize("hq,hkv,n", [(8, 1, 8), (8, 1, 9), (4, 2, 5), (6, 3, 11), (12, 4, 2), (4, 4, 3), (24, 12, 3)])
def test_prefill_attention_ping_pong_short_sequences(torch_cuda, kv, hq, hkv, n):
    """Kv heads that leave XCDs to split, and at least as many sequences as tiles: the
    sequences are spread over the XCDs, also where their number is no multiple of
    the split; and one fewer of them than the split (its tiles are spread, from a
    slot that turns with the sequence)."""
    say(f"prefill ping-pong short kv={kv} hq={hq} hkv={hkv} n={n}")
    split = next(s for s in (1, 2, 4, 8) if hkv * s % 8 == 0)
    for count in {n, split - 1} - {0}:
        segs = [((37 * i) % 90, 1 + (29 * i + 1) % 31) for i in range(count)]
        segs[0] = (5, 2)  # decode rows are single tokens: every segment prefills
        segs = [(s, max(2, m)) for s, m in segs]
        check_segments(torch_cuda, segs, 64, kv, 16, hq, hkv, 2)


@pytest.mark.parametrize("D,kv,hq,hkv,n,rows", [
    (64, "fp16", 2, 2, 130, 33), (64, "int8", 8, 8, 20, 513), (64, "fp16", 16, 4, 40, 70), (64, "fp16", 32, 4, 40, 70),
    (128, "fp16", 4, 4, 40, 129), (128, "int8", 4, 4, 140, 20), (128, "fp16", 8, 4, 21, 160),
    (128, "fp16", 8, 2, 70, 17)])
def test_prefill_attention_rule(torch_cuda, D, kv, hq, hkv, n, rows):
    """The rule's choice (whatever it is) on both sides of its lines: one head per kv
    head, prompts of a whole workgroup of the load-to-LDS kernel, counts around half
    the chip."""
    say(f"prefill rule D={D} kv={kv} hq={hq} hkv={hkv} n={n} rows={rows}")
    segs = [((11 * i) % 50, rows if i == 0 else 2 + (7 * i) % (rows - 1)) for i in range(n)]
    check_segments(torch_cuda, segs, D, kv, 16, hq, hkv, 1)
