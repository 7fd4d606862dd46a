"""How the prefill attention's workgroups go over the eight XCDs (csrc/kernels/attention_prefill.hip)."""
import random

import pytest

from llm_weighted_consensus_amd import ops


def _loads(lens, Hq, Hkv, D):
    """Work of each XCD, and that every (sequence, query head, row tile) has one workgroup: the kernel's own arithmetic."""
    n, most = len(lens), max(lens)
    tile, parts = ops.kernels().prefill_plan(n, sum(lens), most, Hq, Hkv, D)
    group, tiles = Hq // Hkv, -(-most // tile)
    per = -(-tiles * group // parts)
    seen, work = set(), [0] * 8
    for y in range(-(-n * Hkv * parts // 8)):
        for x in range(8 * per):
            share = y * 8 + (x & 7)
            unit, at = share // parts, (x >> 3) * parts + share % parts
            if unit >= n * Hkv or at >= tiles * group:
                continue
            seq, head, t = unit // Hkv, (unit + unit // Hkv) % Hkv * group + at % group, at // group
            assert (seq, head, t) not in seen
            seen.add((seq, head, t))
            if t * tile < lens[seq]:
                work[x & 7] += (t + 1) * min(tile, lens[seq] - t * tile)
    assert len(seen) == n * Hq * tiles
    return work


@pytest.mark.parametrize("Hq,Hkv", [(32, 1), (8, 1), (32, 2), (16, 4), (32, 4), (32, 8), (12, 12), (9, 9), (33, 11)])
@pytest.mark.parametrize("lens", [[8192], [2048, 1500], [4096] + [60] * 30, [500, 400, 300, 200, 100], [256] * 40])
def test_no_xcd_takes_much_more_than_its_share(Hq, Hkv, lens):
    """Few key heads, counts of them that are no multiple of eight, one long prompt among short ones."""
    work = _loads(lens, Hq, Hkv, 128 if Hq == 32 else 64)
    assert max(work) <= 1.25 * sum(work) / 8


def test_every_workgroup_once():
    rng = random.Random(4)
    for _ in range(200):
        Hkv = rng.randint(1, 17)
        lens = [rng.randint(1, rng.choice([3, 70, 300, 2000])) for _ in range(rng.randint(1, 12))]
        _loads(lens, Hkv * rng.randint(1, 8), Hkv, rng.choice([32, 64, 128]))
