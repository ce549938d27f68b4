"""The GEMM's tile geometries at the sizes where they can go wrong: token and row remainders, row blocks
past the last descriptor row, k-groups with unequal (or no) super-blocks, split and unsplit tiles,
mixed types inside a workgroup, x rows further apart than 32-bit offsets reach.  Which geometry a case
runs is asserted (ops.gemm_pick; the sizes are for 256 compute units).  Against the fp64
product of the oracle's weights: bf16 keeps eight bits, so rounding to nearest moves a value by at most
2^-8 of it; one rounding of each weight and of y moves an output by at most 2^-8 (sum |x w| + |y|), fp32
accumulation by far less (the 1 %); over all outputs the error is under 1e-2."""
import numpy as np
import pytest
import torch

from oracle import ggml_ref as G

pytestmark = pytest.mark.gpu


def _close(y, x, wf, bias=None):
    x, wf, y = (np.asarray(v, np.float64) for v in (x, wf, y))
    b = 0.0 if bias is None else np.asarray(bias, np.float64)[None]
    ref, mag = x @ wf.T + b, np.abs(x) @ np.abs(wf).T
    err = np.abs(y - ref)
    return bool((err <= 2.0 ** -8 * (1.01 * mag + 1.01 * np.abs(ref)) + 1e-30).all()) and \
        np.linalg.norm(err) <= 1e-2 * np.linalg.norm(ref)


def _layer(dev, shards, K, seed, cus=0):
    import gguf_hip

    rng = np.random.default_rng(seed)
    raws = [G.make_weights(rng, n, K, wt) for wt, n in shards]
    wf = np.concatenate([G.dequantize(r, wt) for r, (wt, _) in zip(raws, shards)])
    return gguf_hip.pack_layer([torch.from_numpy(r).to(dev) for r in raws], [n for _, n in shards],
                               [wt for wt, _ in shards], cus=cus), wf


def _pick(gl, M):
    from gguf_hip import ops

    i = ops._pick_plan(gl.plans, M)
    info = ops.GqkPlanInfo.from_tuple(gl.plans[i * ops._NPLAN:][:ops._NPLAN])
    return info, ops.gemm_pick(info, M)


def _check(gl, x, wf, bias):
    """y of the layer (wf: its fp64 weights on the GPU) against its bound, three bit-identical repeats, and
    the counters back at zero."""
    import gguf_hip

    y = gguf_hip.mul_mat_grouped(x, gl, bias)
    ref = x.double() @ wf.T + bias.double()
    bound = 2.0 ** -8 * (x.double().abs() @ wf.abs().T + ref.abs())
    worst = float(((y.double() - ref).abs() / (bound + 1e-30)).max())
    print("error over its bound", worst, flush=True)
    assert worst <= 1.01 and float((y.double() - ref).norm()) <= 1e-2 * float(ref.norm())
    for _ in range(3):
        assert torch.equal(gguf_hip.mul_mat_grouped(x, gl, bias), y)
    torch.cuda.synchronize()
    assert int(gl.workspace[:65536].abs().sum()) == 0


def _random_layer(dev, ns, types, K):
    import gguf_hip
    from gguf_hip.synth import random_shard

    raws = [random_shard(n, K, t, dev, seed=t) for n, t in zip(ns, types)]
    wf = torch.cat([gguf_hip.dequantize(w, t, (n, K)) for w, n, t in zip(raws, ns, types)]).double()
    return gguf_hip.pack_layer(raws, ns, list(types)), wf


@pytest.mark.parametrize("shards,nbk", [
    ([(G.Q4_K, 1)], 1),                                     # one row, fewer super-blocks than k-groups
    ([(G.Q3_K, 97)], 2),
    ([(G.Q6_K, 161), (G.IQ3_S, 31)], 3),                    # descriptor rows of different types
    ([(G.Q8_0, 330)], 5),
    ([(G.IQ4_XS, 640), (G.Q2_K, 70), (G.Q5_0, 129)], 7),
    ([(G.Q5_K, 2100)], 9),
    ([(G.IQ4_NL, 33), (G.Q4_0, 64)], 13),
    ([(G.Q4_K, 1097)], 4),                                  # unsplit: eights of tiles and a rest, dealt to XCDs
])
def test_geometries(dev, shards, nbk):
    """Layers up to 2,100 rows: the 64 x 64 geometry, unsplit and split, against the oracle."""
    import gguf_hip

    K = 256 * nbk
    gl, wf = _layer(dev, shards, K, nbk)
    bias = torch.randn(gl.n_total, device=dev).to(torch.bfloat16)
    for M in (33, 63, 64, 65, 97, 128, 129, 255, 257):
        print(shards, nbk, M, flush=True)
        x = torch.randn(M, K, generator=torch.Generator().manual_seed(M)).to(torch.bfloat16)
        y = gguf_hip.mul_mat_grouped(x.to(dev), gl, bias)
        assert _close(y.float().cpu().numpy(), x.float().numpy(), wf, bias.float().cpu().numpy()), M
        for _ in range(2):
            assert torch.equal(gguf_hip.mul_mat_grouped(x.to(dev), gl, bias), y), M
    torch.cuda.synchronize()
    assert int(gl.workspace[:65536].abs().sum()) == 0


@pytest.mark.parametrize("geo,split,n0,nbk,M", [
    ((2, 2, 4), False, 3, 1, 33), ((2, 2, 4), False, 3, 5, 33), ((2, 2, 4), True, 3, 9, 33),
    ((2, 4, 4), False, 3, 3, 761), ((2, 4, 4), False, 3, 7, 761), ((2, 4, 4), True, 3, 20, 221),
    # five waves of row blocks: a workgroup straddles descriptor rows, so its waves decode different types
    ((2, 5, 3), False, 3, 3, 851), ((2, 5, 3), False, 2900, 1, 33), ((2, 5, 3), False, 2900, 5, 33),
    ((4, 4, 2), False, 3, 1, 761), ((4, 4, 2), False, 3, 3, 941), ((4, 4, 2), True, 3, 20, 761),
    ((4, 5, 2), False, 3, 1, 1481), ((4, 5, 2), False, 3, 3, 1481), ((4, 5, 2), True, 3, 20, 851),
    ((8, 8, 1), False, 600, 20, 760),   # remainder tiles only, each shared by several workgroups
    ((8, 8, 1), False, 800, 1, 1801),   # whole tiles dealt to the workgroups, then remainder tiles of one super-block
    ((8, 8, 1), False, 3, 12, 1841),
])
def test_mixed_layers_on_every_geometry(dev, geo, split, n0, nbk, M):
    """A layer with a ragged shard of each type (the mixed-type build), fewer super-blocks than k-groups,
    k-groups of unequal length, split tiles."""
    ns, K = [n0 + 7 * i for i in range(len(G.ALL_TYPES))], 256 * nbk
    gl, wf = _random_layer(dev, ns, G.ALL_TYPES, K)
    info, p = _pick(gl, M)
    assert info.types_mask == 0 and (p["mb"], p["nr"], p["wk"]) == geo and (p["split"] > 1) == split, p
    assert geo[0] < 8 or p["slots"] > 0, p
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(M)).to(torch.bfloat16).to(dev)
    print(geo, p, flush=True)
    _check(gl, x, wf, torch.randn(gl.n_total, device=dev).to(torch.bfloat16))


@pytest.mark.parametrize("geo,split,n,nbk,M", [
    ((2, 2, 4), False, 97, 5, 34), ((2, 2, 4), True, 97, 9, 34), ((2, 4, 4), False, 257, 5, 2111),
    ((2, 4, 4), True, 33, 20, 1391), ((2, 5, 3), False, 33000, 4, 33), ((4, 4, 2), False, 20600, 3, 72),
    ((4, 4, 2), True, 257, 20, 2111), ((4, 5, 2), False, 16500, 3, 131), ((4, 5, 2), True, 16500, 20, 72),
    ((8, 8, 1), False, 24700, 3, 401),
])
def test_each_type_on_every_geometry(dev, geo, split, n, nbk, M):
    """The single-type builds: the barrier's count of loads in flight depends on the geometry and on the
    type's loads."""
    K = 256 * nbk
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(M)).to(torch.bfloat16).to(dev)
    for t in G.ALL_TYPES:
        gl, wf = _random_layer(dev, [n], [t], K)
        info, p = _pick(gl, M)
        assert info.types_mask == t and (p["mb"], p["nr"], p["wk"]) == geo and (p["split"] > 1) == split, p
        assert geo[0] < 8 or p["slots"] > p["tail_wgs"], p
        print(G.NAMES[t], p, flush=True)
        _check(gl, x, wf, torch.randn(n, device=dev).to(torch.bfloat16))


def _launches(fn):
    """fn()'s result and how many kernels of the linear forms it launched."""
    torch.cuda.synchronize()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        y = fn()
        torch.cuda.synchronize()
    return y, sum("gemm_kernel" in e.name or "gemv" in e.name for e in prof.events())


@pytest.mark.parametrize("ldx", [1 << 22, (1 << 22) + 8, (1 << 27) + 64])
def test_rows_far_apart(dev, ldx):
    """Row strides of x at the last one that 32-bit byte offsets from a tile's first row serve (8 MiB), just
    above it, and where such offsets would wrap within 32 rows: one launch each, the same bits as from a
    contiguous x, in the mid form (slab and split), the GEMM (split) and the 256 x 256 form."""
    import gguf_hip

    K = 512
    small, wf = _layer(dev, [(G.Q4_K, 130), (G.IQ3_S, 64)], K, 3)
    slab, _ = _layer(dev, [(G.Q4_K, 130), (G.IQ3_S, 64)], K, 3, cus=8)
    wide = None
    if ldx < 1 << 23:
        wide, _ = _random_layer(dev, [800 + 7 * i for i in range(len(G.ALL_TYPES))], G.ALL_TYPES, K)
        assert _pick(wide, 1801)[1]["mb"] == 8
    for gl, M in ((small, 3), (small, 18), (slab, 32), (small, 34), (small, 41), (wide, 1801)):
        if gl is None:
            continue
        x = torch.empty((M - 1) * ldx + K, dtype=torch.bfloat16, device=dev).as_strided((M, K), (ldx, 1))
        x.copy_(torch.randn(M, K, generator=torch.Generator().manual_seed(M)).to(torch.bfloat16))
        print(ldx, M, flush=True)
        y, count = _launches(lambda: gguf_hip.mul_mat_grouped(x, gl))
        assert count == 1, (M, count)
        assert torch.equal(y, gguf_hip.mul_mat_grouped(x.contiguous(), gl)), M
        if gl is not wide:
            assert _close(y.float().cpu().numpy(), x.float().cpu().numpy(), wf), M
        del x
