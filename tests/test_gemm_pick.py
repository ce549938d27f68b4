"""The GEMM's choice of tile geometry, on the host (256 compute units)."""
import random

import pytest

from oracle import ggml_ref as G

CUS = 256


def _pick(ns, K, M, wt=G.Q4_K):
    from gguf_hip import ops

    shards, off = [], 0
    for n in ns:
        shards.append((wt, n, off))
        off += ops.tiles_bytes(wt, n, K)
    bucket = next((m for m in ops.GEMM_PLAN_M if M <= m), ops.GEMM_PLAN_M[-1])
    info, _ = ops.plan(shards, K, bucket, 0, CUS)
    return info, ops.gemm_pick(info, M, CUS)


@pytest.mark.parametrize("n,K,M", [(33024, 5120, 384), (24778, 1280, 563), (24140, 256, 564), (18043, 512, 1094),
                                   (8919, 256, 2046), (33348, 4352, 375)])
def test_a_short_remainder_counts_as_the_round_it_takes(n, K, M):
    """Layers whose 256 x 256 tiles leave a few past whole rounds of the CUs: these take few workgroups, so
    the tail lasts like a round, and 128-token tiles are measured 1.05-2.5 times as fast."""
    assert _pick([n], K, M)[1]["mb"] == 4


def test_picks_are_consistent():
    """Every pick covers the layer, splits only what fits the CUs at once, and its partials fit the
    workspace that serves every GEMM plan (2 x CUs - 2 slots of 256 KiB)."""
    rng, seen = random.Random(7), set()
    for _ in range(1500):
        ns = [1 + int(36000 ** rng.random()) for _ in range(rng.choice((1, 1, 2, 3)))]
        K, M = 256 * (1 + int(68 ** rng.random())), 33 + int(8000 ** rng.random())
        info, p = _pick(ns, K, M)
        seen.add((p["mb"], p["nr"], p["wk"]))
        per, nb = 8 if info.bm == 256 else 4, K // 256
        tiles = -(-info.n_desc * per // p["nr"]) * -(-M // (32 * p["mb"]))
        if p["mb"] == 8:
            assert info.bm == 256 and p["split"] == 1 and p["wgs"] == (CUS if tiles >= CUS else p["tail_wgs"])
            assert p["slots"] == (tiles % CUS + p["tail_wgs"] - 1 if tiles % CUS else 0)
            assert 1 <= p["tail_wgs"] <= CUS and p["slots"] <= 2 * CUS - 2
        else:
            assert p["wgs"] == tiles * p["split"] and 1 <= p["split"] <= max(1, nb // p["wk"])
            assert p["slots"] == (p["wgs"] if p["split"] > 1 else 0) and (p["split"] == 1 or p["wgs"] <= CUS)
    assert seen == {(2, 2, 4), (2, 4, 4), (2, 5, 3), (4, 4, 2), (4, 5, 2), (8, 8, 1)}
