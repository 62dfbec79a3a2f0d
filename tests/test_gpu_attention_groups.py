"""Attention of prefills and chunks with one, two and four key groups a block and with split keys, at the edges of
their tiles: rows next to a tile, step or block boundary against the oracle, every row finite."""
import numpy as np
import pytest

from gpu_util import announce, check_band
from test_gpu_parity import run_attention

pytestmark = pytest.mark.gpu

D = 128


def _edge_rows(B, S, start, Hq, Hkv):
    """Rows of the first and last positions and of those around multiples of 16, 32 and 64 keys and columns."""
    G = Hq // Hkv
    pos = {0, 1, S - 2, S - 1}
    for edge in (32, 64, 128, 256):
        pos |= {edge - start - 1, edge - start, edge // G - 1, edge // G, edge - 1, edge, 3 * edge // G}
    pos |= {(start + S) // 128 * 128 - start - 1, (start + S) // 128 * 128 - start, S // 2, 2 * S // 3}
    pos = sorted(p for p in pos if 0 <= p < S)
    heads = sorted({0, G - 1, G, Hq - 1} & set(range(Hq)))
    batches = sorted({0, B - 1})
    return np.array([(b * S + s) * Hq + h for b in batches for s in pos for h in heads])


# four groups (few blocks): one step or less, odd remainders, a group without a tile, G = 1, 5, 32;
# two groups (257 .. 512 blocks of 128 columns); one group; chunks that stay whole
@pytest.mark.parametrize("B,S,start,Hq,Hkv", [
    (1, 2, 0, 16, 8), (1, 65, 0, 8, 8), (1, 97, 0, 32, 8), (2, 129, 0, 10, 2), (1, 161, 3, 32, 1), (1, 300, 20, 40, 8),
    (1, 1023, 0, 4, 1), (2, 130, 255, 16, 8), (1, 1500, 0, 32, 8), (2, 1001, 0, 32, 8), (1, 1750, 31, 32, 8),
    (2, 1025, 0, 40, 8), (1, 64, 0, 32, 8), (1, 33, 31, 16, 8)])
def test_gqa_attention_key_groups(q3k, hip, oracle, synth, B, S, start, Hq, Hkv):
    name = f"gqa_attention groups B={B} S={S} start={start} Hq={Hq} Hkv={Hkv}"
    announce(name)
    cap = start + S + 5
    q = synth.normal_bf16(180, S, (B, S, Hq * D))
    k = synth.normal_bf16(181, S, (B, cap, Hkv, D))
    v = synth.normal_bf16(182, S, (B, cap, Hkv, D))
    got = run_attention(q3k, hip, q, k, v, B, S, Hq, start)
    rows = _edge_rows(B, S, start, Hq, Hkv)
    prim, lo, hi = oracle.gqa_attention(q, k[:, :start + S], v[:, :start + S], Hq, start, rows=rows)
    check_band(oracle, name, got.reshape(-1, D)[rows], prim, lo, hi)
    assert np.isfinite(synth.bf16_to_f32(got)).all()


# chunks and prefills whose keys are split: slices that some query blocks do not reach, blocks with a single slice
# (which write their result themselves); rows merged by a block each (few), by 16 lanes (many, of few slices) and by a
# wave (many, of more: 9, 16 and, in two rounds, 22 slices)
@pytest.mark.parametrize("B,S,start,Hq,Hkv", [
    (1, 2048, 0, 4, 1), (1, 7, 4090, 32, 8), (1, 70, 4000, 32, 8), (1, 260, 4000, 32, 8), (1, 600, 3000, 5, 1),
    (1, 3000, 0, 2, 1), (1, 2, 8000, 8, 1), (1, 1075, 0, 2, 1), (1, 167, 11748, 16, 8), (1, 701, 11748, 4, 1)])
def test_gqa_attention_key_groups_split(q3k, hip, oracle, synth, B, S, start, Hq, Hkv):
    name = f"gqa_attention groups, split, B={B} S={S} start={start} Hq={Hq} Hkv={Hkv}"
    announce(name)
    cap = start + S
    q = synth.normal_bf16(183, S, (B, S, Hq * D))
    k = synth.normal_bf16(184, S, (B, cap, Hkv, D))
    v = synth.normal_bf16(185, S, (B, cap, Hkv, D))
    got = run_attention(q3k, hip, q, k, v, B, S, Hq, start, split=True)
    rows = _edge_rows(B, S, start, Hq, Hkv)
    prim, lo, hi = oracle.gqa_attention(q, k, v, Hq, start, rows=rows)
    check_band(oracle, name, got.reshape(-1, D)[rows], prim, lo, hi)
    assert np.isfinite(synth.bf16_to_f32(got)).all()


# at most 32 columns a pair (decode): one, two and four waves a block; fewer keys than one tile, waves without a
# tile, partial tiles; several positions; slices of one wave and of several; more sequences than one round holds
@pytest.mark.parametrize("B,S,start,Hq,Hkv,split", [
    (1, 1, 0, 16, 8, False), (3, 1, 31, 32, 8, False), (2, 1, 32, 40, 8, False), (1, 1, 127, 32, 1, False),
    (1, 1, 200, 32, 8, False), (2, 3, 250, 40, 8, False), (1, 8, 90, 32, 8, False), (40, 1, 161, 32, 8, False),
    (65, 1, 100, 32, 8, False), (1, 1, 2100, 16, 8, False), (1, 1, 700, 16, 8, True), (2, 4, 1500, 32, 8, True),
    (1, 1, 9000, 5, 1, True), (5, 1, 3001, 8, 8, True), (20, 1, 2500, 4, 2, True)])
def test_gqa_attention_decode_waves(q3k, hip, oracle, synth, B, S, start, Hq, Hkv, split):
    name = f"gqa_attention decode waves B={B} S={S} start={start} Hq={Hq} Hkv={Hkv} split={split}"
    announce(name)
    cap = start + S + 3
    q = synth.normal_bf16(186, B, (B, S, Hq * D))
    k = synth.normal_bf16(187, B, (B, cap, Hkv, D))
    v = synth.normal_bf16(188, B, (B, cap, Hkv, D))
    got = run_attention(q3k, hip, q, k, v, B, S, Hq, start, split=split)
    rows = np.unique(np.concatenate([np.arange(min(B, 3) * S * Hq), np.arange((B - 1) * S * Hq, B * S * Hq)]))
    prim, lo, hi = oracle.gqa_attention(q, k[:, :start + S], v[:, :start + S], Hq, start, rows=rows)
    check_band(oracle, name, got.reshape(-1, D)[rows], prim, lo, hi)
    assert np.isfinite(synth.bf16_to_f32(got)).all()
