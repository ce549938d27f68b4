"""The dequantizers and the repack where their wide accesses could go wrong: rows at odd addresses and
strides, rows shorter than a workgroup's span, partial 64-row tiles, one super-block, output rows that
take no 16-byte stores.  Bit-exact against the oracle."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import ggml_ref as G

pytestmark = pytest.mark.gpu


def _odd_view(raw, dev, shift, pad):
    """raw's rows at byte `shift` of a buffer, `pad` bytes between rows."""
    n, b = raw.shape
    buf = torch.full((shift + n * (b + pad),), 0xA5, dtype=torch.uint8, device=dev)
    v = buf.as_strided((n, b), (b + pad, 1), shift)
    v.copy_(torch.from_numpy(raw).to(dev))
    return v


@pytest.mark.parametrize("wt", G.ALL_TYPES)
def test_edges(dev, wt):
    import gguf_hip
    from gguf_hip import _lib

    rng = np.random.default_rng(wt)
    small = [32, 96, 1056] if G.TYPES[wt][1] == 32 else []
    for K in small + [256, 512, 8448, 9216]:
        for n, shift, pad in ((1, 0, 0), (3, 1, 1), (65, 2, 0), (70, 3, 5), (64, 8, 8)):
            raw = G.random_blocks(rng, n, K, wt)
            W = _odd_view(raw, dev, shift, pad)
            ref = G.dequantize(raw, wt, K)
            f32 = torch.from_numpy(ref)
            want = {torch.float32: f32, torch.bfloat16: f32.to(torch.bfloat16), torch.float16: f32.to(torch.float16)}
            for dt, w in want.items():
                bits = torch.int32 if dt == torch.float32 else torch.int16
                got = gguf_hip.ggml_dequantize(W, wt, n, K, dt)
                assert torch.equal(got.cpu().view(bits), w.view(bits)), (K, n, shift, dt)
                code = {torch.float32: 0, torch.bfloat16: 1, torch.float16: 2}[dt]
                out = torch.zeros(n, K + 1, dtype=dt, device=dev)   # odd row stride
                st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
                _lib.check(_lib.lib.gqk_dequantize(W.data_ptr(), W.stride(0), wt, n, K, out.data_ptr(), K + 1, code, st), "dq")
                assert torch.equal(out[:, :K].cpu().contiguous().view(bits), w.view(bits)) and not out[:, K].any()
                if K % 256 == 0:
                    tiles = gguf_hip.repack_tiles(W, n, wt)
                    assert torch.equal(gguf_hip.dequantize_tiles(tiles, n, K, wt, dt).cpu().view(bits), w.view(bits))
                    out.zero_()
                    _lib.check(_lib.lib.gqk_dequantize_tiles(tiles.data_ptr(), wt, n, K, out.data_ptr(), K + 1, code, st), "dq")
                    assert torch.equal(out[:, :K].cpu().contiguous().view(bits), w.view(bits)) and not out[:, K].any()
            if K % 256 == 0:
                assert np.array_equal(gguf_hip.unrepack_tiles(tiles, n, K, wt).cpu().numpy(), raw), (K, n, shift)
                one = gguf_hip.repack_tiles(torch.from_numpy(raw).to(dev), n, wt)
                assert torch.equal(one, tiles), (K, n, shift)   # the tiles do not depend on where the rows lay
