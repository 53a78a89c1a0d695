"""Every form of the 16-bit prefill kernels that the launch rules choose among, reached by wide
models' small prompts: pairs of row blocks per KV head with each group size and one or two
teams of waves, their second segment of page ids, and one key tile for two row blocks.
test_launch_rules.py checks, without a GPU, that these shapes take the forms they name."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import HD, THETA, from_dev, make_tables, normal, to_dev
from test_gpu_decode import check

pytestmark = pytest.mark.gpu
KVS = {"f16": 1, "f16split": 1, "bf16": 2}

# (rows, query heads, KV heads): two teams, then one, of 1 to 8 waves (query heads per KV head).
PAIRS_TWO_TEAMS = [(111, 43 * g, 43) for g in range(1, 9)]
PAIRS_ONE_TEAM = [(175, 43 * g, 43) for g in range(1, 9)]
# (first position, rows, heads, KV heads): the rows' keys run past 32,768 (512 tiles).
SEGMENTS_TWO_TEAMS, SEGMENTS_ONE_TEAM = (32300, 700, 8, 8), (31900, 1060, 8, 8)
ONE_TILE_OF_TWO_BLOCKS = (20, 320, 40)


@pytest.fixture
def rounding(ie, kv):
    prev = ie.set_prefill_rounding(ie.PREFILL_SPLIT if kv == "f16split" else ie.PREFILL_SINGLE)
    yield
    ie.set_prefill_rounding(prev)


def prefill(ie, dev, q, kp, vp, kvt, row_pos, row_seq, tables, nh, nkv):
    out = torch.full(q.shape, float("nan"), device=dev)
    ie.attention_prefill(out, to_dev(q, dev), to_dev(kp, dev, kvt), to_dev(vp, dev, kvt),
                         to_dev(row_pos, dev), to_dev(row_seq, dev), to_dev(tables, dev),
                         tables.shape[1], nh, nkv, HD)
    torch.cuda.synchronize()
    return from_dev(out)


@pytest.mark.parametrize("T,nh,nkv", PAIRS_TWO_TEAMS + PAIRS_ONE_TEAM)
@pytest.mark.parametrize("kv", list(KVS))
def test_pairs(ie, O, dev, kv, rounding, T, nh, nkv):
    """A prompt that starts mid-tile, as the second of two sequences, with NaN in every row of
    the pool that its positions do not hold and two pages of its context outside the pool
    (expected: attention over the sequence without those 32 positions); then the same rows
    appended and attended in one call, bit for bit as by rope_and_cache + attention_prefill."""
    kvt = KVS[kv]
    rng = np.random.default_rng(T + nh)
    start = 77
    n, kvd = start + T, nkv * HD
    tables, max_pages, num_pages = make_tables([50, n], rng, extra_pages=3)
    at = tables[1, np.arange(n) // 16] * 16 + np.arange(n) % 16
    kp, vp = (np.full((num_pages * 16, kvd), 0x7FFF, np.uint16) for _ in range(2))
    k, v = (O.round_to_kv(normal(rng, (n, kvd)), kvt) for _ in range(2))
    kp[at], vp[at] = k, v
    row_pos, row_seq = np.arange(start, n, dtype=np.int32), np.ones(T, np.int32)
    q = normal(rng, (T, nh * HD))
    holes = tables.copy()
    holes[1, 1:3] = num_pages + 7, -3  # positions 16 .. 47
    keep = np.r_[0:16, 48:n]
    kc, vc = (O.widen_kv(a[keep], kvt).reshape(-1, kvd) for a in (k, v))
    want = O.attention(q, kc, vc, start - 32, nh, nkv, HD, threads=8)
    check(O, prefill(ie, dev, q, kp, vp, kvt, row_pos, row_seq, holes, nh, nkv), want, kvt)

    table = ie.rope_table(n, HD, THETA).to(dev)
    rows = (to_dev(row_pos, dev), to_dev(row_seq, dev), to_dev(tables, dev), max_pages, nh, nkv, HD)
    dk, dv = to_dev(normal(rng, (T, kvd)), dev), to_dev(normal(rng, (T, kvd)), dev)
    outs, pools = [], []
    for fused in (True, False):
        dq, pk, pv = to_dev(q, dev), to_dev(kp, dev, kvt), to_dev(vp, dev, kvt)
        out = torch.full(q.shape, float("nan"), device=dev)
        if fused:
            ie.rope_cache_attention_prefill(out, dq, dk, dv, pk, pv, table, *rows)
        else:
            ie.rope_and_cache(dq, dk, dv, pk, pv, table, *rows)
            ie.attention_prefill(out, dq, pk, pv, *rows)
        outs.append(out)
        pools.append((pk, pv))
    torch.cuda.synchronize()
    assert torch.equal(outs[0].view(torch.int32), outs[1].view(torch.int32))
    assert all(torch.equal(a.view(torch.int16), b.view(torch.int16)) for a, b in zip(*pools))
    assert torch.isfinite(outs[0]).all()


@pytest.mark.parametrize("start,T,nh,nkv", [SEGMENTS_TWO_TEAMS, SEGMENTS_ONE_TEAM])
@pytest.mark.parametrize("kv", list(KVS))
def test_second_segment_of_page_ids(ie, O, dev, kv, rounding, start, T, nh, nkv):
    """Rows on both sides of position 32,768."""
    kvt = KVS[kv]
    rng = np.random.default_rng(T)
    n = start + T
    tables, max_pages, num_pages = make_tables([n], rng)
    kp, vp = (O.round_to_kv(normal(rng, (num_pages * 16, nkv * HD)), kvt) for _ in range(2))
    row_pos, row_seq = np.arange(start, n, dtype=np.int32), np.zeros(T, np.int32)
    q = normal(rng, (T, nh * HD))
    rows = np.unique(np.r_[0, 32767 - start, 32768 - start, 32768 - start + 64, T // 2, T - 17, T - 1])
    want = O.paged_attention(q[rows], kp, vp, kvt, row_pos[rows], row_seq[rows], tables, max_pages, nh,
                             nkv, HD, threads=8)
    check(O, prefill(ie, dev, q, kp, vp, kvt, row_pos, row_seq, tables, nh, nkv)[rows], want, kvt)


@pytest.mark.parametrize("kv", list(KVS))
@pytest.mark.parametrize("bad", [0.0, np.inf])
def test_one_tile_of_two_blocks(ie, O, dev, kv, rounding, bad):
    """20 rows on an empty cache: one 32-key tile, finished by the wave that takes it; an
    infinite value at position 18 does not reach rows 0 to 15."""
    T, nh, nkv = ONE_TILE_OF_TWO_BLOCKS
    kvt = KVS[kv]
    rng = np.random.default_rng(nh)
    tables, max_pages, num_pages = make_tables([T], rng)
    kp, vp = (O.round_to_kv(normal(rng, (num_pages * 16, nkv * HD)), kvt) for _ in range(2))
    row_pos, row_seq = np.arange(T, dtype=np.int32), np.zeros(T, np.int32)
    q = normal(rng, (T, nh * HD))
    want = O.paged_attention(q, kp, vp, kvt, row_pos, row_seq, tables, max_pages, nh, nkv, HD, threads=8)
    clean = np.ones(want.shape, bool)
    if bad:
        vp[tables[0, 1] * 16 + 2, 3] = O.round_to_kv(np.array([bad], np.float32), kvt)[0]
        clean[16:, 3:nh // nkv * HD:HD] = False
    got = prefill(ie, dev, q, kp, vp, kvt, row_pos, row_seq, tables, nh, nkv)
    check(O, np.where(clean, got, 0), np.where(clean, want, 0), kvt)
