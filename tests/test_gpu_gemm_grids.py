"""Prefill GEMM grids (wq_gemm.hip): row counts at the edges of the 64- and
128-row tiles on each grid give the rows of the 64-wide grid bit for bit (one
k order on every grid), the fused epilogues equal the plain GEMM plus the
elementwise op, and sampled rows hold the oracle's bar (``parity_ok``)."""
import numpy as np
import pytest
import torch

from oracle import qdq, synth
from ondeviceinfer_amd import _native
from ondeviceinfer_amd.weight_quantization import backend as wq

pytestmark = pytest.mark.gpu


# (m, n, k), one tile height after the other: 2 tiles x 80 rows (129; 673 =
# 8 x 80 + 33), 4 x 96 (448 ends inside a block, 34800 inside a slice; 577 =
# 6 x 96 + 1), 4 x 112 (777, 785 takes 128), 2 x 96 (1056 = 11 x 96), 2 x 128
# (1345, 1500; 5112 ends inside a tile), 1 x 64, 2 x 64, 4 x 64.
SHAPES = [(129, 34816, 256), (673, 7168, 384), (448, 34800, 128), (577, 17400, 256), (777, 34816, 128),
          (785, 34816, 128), (1056, 5112, 256), (1345, 5120, 384), (1500, 5112, 256), (200, 5120, 640),
          (449, 4040, 256), (700, 5120, 256)]


def same(a, b):
    torch.cuda.synchronize()
    return torch.equal(a.view(torch.int16), b.view(torch.int16))


def rows_of(m):
    return np.array(sorted({r for r in (0, 63, 64, 127, 128, m - 2, m - 1) if 0 <= r < m}))


def check(y, x, w32, label):
    rows = rows_of(y.shape[0])
    torch.cuda.synchronize()
    expected = (x.cpu().numpy()[rows].astype(np.float32) @ w32.T).astype(np.float16)
    metrics = qdq.parity_metrics(y.cpu().numpy()[rows], expected)
    assert qdq.parity_ok(metrics), (label, metrics)


@pytest.mark.parametrize('m,n,k', SHAPES)
@pytest.mark.parametrize('fmt', ['w4', 'int8'])
def test_grids_agree_and_hold_the_oracle(gpu, fmt, m, n, k):
    print(f'[grid] {fmt} m={m} n={n} k={k}', flush=True)
    gen = torch.Generator(device=gpu).manual_seed(m + n)
    x = torch.randn(m, k, generator=gen, device=gpu).half()
    res = torch.randn(m, n, generator=gen, device=gpu).half()
    if fmt == 'w4':
        weights, _ = synth.w4_case(n, k, 1, seed=n % 83 + k, name='p.weight')
        layer = {key: torch.from_numpy(np.ascontiguousarray(v)).to(gpu) for key, v in weights.items()}
        wq.CompressedLinearBackend('marlin', group_size=128).prepare(layer, 'p.weight')
        p = layer['p._prepared']
        w32 = qdq.decode_weight(weights, 'p.weight', group_size=128).astype(np.float32)
        plain = lambda a: _native.w4a16_linear(a, p.tiles, p.meta, n, 128)
        fused = lambda mode, r=None: _native.w4a16_linear_epilogue(x, p.tiles, p.meta, n, 128, mode, r)
        takes = lambda mode: _native.w4a16_epilogue_supported(m, n, k, 128, mode)
    else:
        _, q, s, _ = synth.int8_case(n, k, 1, seed=n % 83 + k)
        q, s = (torch.from_numpy(v).to(gpu) for v in (q, s))
        tiles = _native.w8_repack(q)
        w32 = qdq.dequantize_linear_weight(q.cpu().numpy(), s.cpu().numpy()).astype(np.float32)
        plain = lambda a: _native.w8a16_linear(a, tiles, s)
        fused = lambda mode, r=None: _native.w8a16_linear_epilogue(x, tiles, s, mode, r)
        takes = lambda mode: _native.w8a16_epilogue_supported(m, n, k, mode)
        assert same(plain(x), _native.w8a16_linear(x, q, s))   # row-major: its own grids
    y = plain(x)
    check(y, x, w32, (fmt, m, n, k))
    # The same rows inside a longer call, which takes the widest grid.
    longer = plain(torch.cat([x, torch.randn(4096 - m, k, generator=gen, device=gpu).half()]))
    assert same(y, longer[:m])
    if takes(_native.EPI_RESIDUAL):
        assert same(fused(_native.EPI_RESIDUAL, res), res + y)
    if takes(_native.EPI_SILU_MUL):
        assert same(fused(_native.EPI_SILU_MUL), _native.silu_mul(y))
