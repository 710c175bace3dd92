"""GPU parity of the 5-to-64-row linears (wq_mid.hip) against the CPU oracle at
the edges of its 16-row chunks, tile groups, stages and splits.

Bars as in test_gpu_parity.py (``oracle.qdq.parity_ok``); the two INT8 layouts
run the same plan and must give the same bits."""
import numpy as np
import pytest
import torch

from oracle import qdq, synth
from ondeviceinfer_amd import _native
from ondeviceinfer_amd.weight_quantization import backend as wq

pytestmark = pytest.mark.gpu

ROWS = (5, 16, 17, 33, 36, 48, 49, 64)   # both ends of the 16-row chunks


def dev(a, device):
    return torch.from_numpy(np.ascontiguousarray(a)).to(device)


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


def check_parity(actual, expected, label):
    m = qdq.parity_metrics(actual, expected)
    print(label, {k: (round(v, 8) if isinstance(v, float) else v) for k, v in m.items()}, flush=True)
    assert qdq.parity_ok(m), (label, m)


# (n, k, group, symmetric): one block (the odd parity idle); a partial last tile
# group (1000 rows = 63 tiles) over 31 blocks, and over 66 with groups of 384 =
# three blocks (stages start inside a group); whole groups of 256 blocks wide;
# 1088 tiles (three splits); 1600 tiles (two splits).
@pytest.mark.parametrize('n,k,g,sym', [(512, 128, 128, False), (1000, 3968, 128, False), (1000, 8448, 384, True),
                                       (2048, 2560, 256, False), (17408, 1280, 128, False),
                                       (25600, 1280, 128, True)])
def test_w4_mid_matches_oracle(gpu, n, k, g, sym):
    name = 'p.weight'
    weights, x = synth.w4_case(n, k, max(ROWS), seed=n % 89 + k, group_size=g, symmetric=sym, name=name)
    layer = {key: dev(v, gpu) for key, v in weights.items()}
    backend = wq.CompressedLinearBackend('marlin', group_size=g)
    backend.prepare(layer, name)
    w32 = qdq.decode_weight(weights, name, group_size=g).astype(np.float32)
    for m in ROWS:
        y = host(backend.linear(dev(x[:m], gpu), layer, name))
        check_parity(y, (x[:m].astype(np.float32) @ w32.T).astype(np.float16), f'w4 mid n={n} k={k} g={g} m={m}')


@pytest.mark.parametrize('n,k', [(512, 128), (1001, 3968), (2050, 8448), (17408, 1280), (34816, 640)])
def test_w8_mid_matches_oracle_in_both_layouts(gpu, n, k):
    _, q, s, x = synth.int8_case(n, k, max(ROWS), seed=n % 97 + k)
    qd, sd = dev(q, gpu), dev(s, gpu)
    tiles = _native.w8_repack(qd)
    w32 = qdq.dequantize_linear_weight(q, s).astype(np.float32)
    bias = (np.random.default_rng(k).standard_normal(n) * 0.1).astype(np.float16)
    for m in ROWS:
        xd = dev(x[:m], gpu)
        y = _native.w8a16_linear(xd, tiles, sd, bias=dev(bias, gpu))
        assert torch.equal(y, _native.w8a16_linear(xd, qd, sd, bias=dev(bias, gpu)))
        expected = (x[:m].astype(np.float32) @ w32.T + bias.astype(np.float32)).astype(np.float16)
        check_parity(host(y), expected, f'w8 mid n={n} k={k} m={m}')


def test_mid_splits_run_on_two_streams_at_once_and_under_capture(gpu):
    """Every call brings its own partials: calls on two streams that overlap,
    and replays of two captured graphs, equal the calls made one by one; a
    workspace too small for the splits runs the skinny kernels within the bar."""
    gen = torch.Generator(device=gpu).manual_seed(3)
    w = wq.CompressedLinearBackend('w8a16')
    layer = {'p.weight': torch.randint(-127, 128, (5120, 5120), generator=gen, device=gpu).to(torch.int8),
             'p.weight_scale': torch.rand(5120, 1, generator=gen, device=gpu) * 1e-3 + 1e-4}
    w.prepare(layer, 'p.weight')
    xs = [torch.randn(40, 5120, generator=gen, device=gpu).half() for _ in range(2)]
    refs = [w.linear(x, layer, 'p.weight').clone() for x in xs]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in xs]
    outs = [[], []]
    for _ in range(8):
        for s, x, o in zip(streams, xs, outs):
            with torch.cuda.stream(s):
                o.append(w.linear(x, layer, 'p.weight'))
    torch.cuda.synchronize()
    for o, ref in zip(outs, refs):
        assert all(torch.equal(y, ref) for y in o)
    graphs, ys = [], []
    for s, x in zip(streams, xs):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            ys.append(w.linear(x, layer, 'p.weight'))
        graphs.append(g)
    for _ in range(3):
        for g, s, y in zip(graphs, streams, ys):
            with torch.cuda.stream(s):
                y.zero_()
                g.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(y, ref) for y, ref in zip(ys, refs))
    p = layer['p._prepared']
    small = _native.w8a16_linear(xs[0], p.qweight, p.scale, workspace=torch.empty(16, dtype=torch.uint8, device=gpu))
    check_parity(host(small), host(refs[0]).astype(np.float32), 'skinny fallback')


@pytest.mark.parametrize('m,n', [(24, 7168), (128, 1024)])
def test_counted_splits_run_on_two_streams_at_once_and_under_capture(gpu, m, n):
    """The W4 splits with arrival counters (24 rows, and the deep-ring GEMM at
    128): calls on two streams that overlap, and replays of two captured graphs
    beside each other and beside eager calls, equal the calls made one by one."""
    weights, _ = synth.w4_case(n, 5120, 1, seed=n + m, name='p.weight')
    layer = {key: dev(v, gpu) for key, v in weights.items()}
    w = wq.CompressedLinearBackend('marlin')
    w.prepare(layer, 'p.weight')
    assert _native.w4a16_workspace_zeroed(m, n, 5120, 128) > 0
    gen = torch.Generator(device=gpu).manual_seed(4)
    xs = [torch.randn(m, 5120, generator=gen, device=gpu).half() for _ in range(2)]
    refs = [w.linear(x, layer, 'p.weight').clone() for x in xs]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in xs]
    outs = [[], []]
    for _ in range(8):
        for s, x, o in zip(streams, xs, outs):
            with torch.cuda.stream(s):
                o.append(w.linear(x, layer, 'p.weight'))
    torch.cuda.synchronize()
    for o, ref in zip(outs, refs):
        assert all(torch.equal(y, ref) for y in o)
    graphs, ys = [], []
    for x in xs:   # both on one capture stream, as torch captures by default
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=streams[0]):
            ys.append([w.linear(x, layer, 'p.weight') for _ in range(3)])
        graphs.append(g)
    for _ in range(4):
        for g, s, y in zip(graphs, streams, ys):
            with torch.cuda.stream(s):
                for t in y:
                    t.zero_()
                g.replay()
        beside = [w.linear(x, layer, 'p.weight') for x in xs]   # on the default stream
        torch.cuda.synchronize()
        for y, b, ref in zip(ys, beside, refs):
            assert torch.equal(b, ref) and all(torch.equal(t, ref) for t in y)


# Shapes the shared-activation kernel does take: an odd block count over a
# partial last tile group (the last stage half empty) in many splits; groups of
# 384 = three blocks (stages start inside a group); ten-tile groups in two
# splits, and unsplit over a partial last group; 33 to 35 rows.
@pytest.mark.parametrize('m,n,k,g', [(5, 1000, 12416, 128), (17, 1000, 12416, 128), (12, 7168, 5120, 128),
                                     (33, 1000, 8448, 384), (34, 7168, 5120, 128), (35, 1024, 5120, 256),
                                     (35, 17408, 2560, 128), (49, 17400, 2432, 128), (64, 5112, 4992, 128),
                                     (8, 25608, 4224, 128), (16, 25600, 3968, 128)])
def test_w4_mid_shapes_match_oracle(gpu, m, n, k, g):
    plan = _native.linear_plan('w4a16', m, n, k)
    print(f'[mid] m={m} n={n} k={k} g={g}: {plan}', flush=True)
    assert plan.startswith('mid')
    weights, x = synth.w4_case(n, k, m, seed=n % 89 + k, group_size=g, name='p.weight')
    layer = {key: dev(v, gpu) for key, v in weights.items()}
    backend = wq.CompressedLinearBackend('marlin', group_size=g)
    backend.prepare(layer, 'p.weight')
    w32 = qdq.decode_weight(weights, 'p.weight', group_size=g).astype(np.float32)
    y = backend.linear(dev(x, gpu), layer, 'p.weight')
    check_parity(host(y), (x.astype(np.float32) @ w32.T).astype(np.float16), plan)
    assert torch.equal(backend.linear(dev(x, gpu), layer, 'p.weight'), y)


# INT8 shapes the kernel takes: both ends of the 16-row chunks, an odd block count, partial last tile groups,
# n not a multiple of 4, many splits, ten-tile groups unsplit and in two splits.
@pytest.mark.parametrize('m,n,k', [(5, 5112, 17280), (16, 1001, 12416), (17, 1000, 8064), (32, 17408, 4992),
                                   (33, 1001, 3968), (48, 34816, 640), (49, 2050, 8448), (64, 17408, 1280)])
def test_w8_mid_shapes_match_oracle_in_both_layouts(gpu, m, n, k):
    plan = _native.linear_plan('w8a16', m, n, k)
    print(f'[mid] int8 m={m} n={n} k={k}: {plan}', flush=True)
    assert plan.startswith('mid')
    _, q, s, x = synth.int8_case(n, k, m, seed=n % 97 + k)
    qd, sd, xd = dev(q, gpu), dev(s, gpu), dev(x, gpu)
    w32 = qdq.dequantize_linear_weight(q, s).astype(np.float32)
    y = _native.w8a16_linear(xd, _native.w8_repack(qd), sd)
    assert torch.equal(y, _native.w8a16_linear(xd, qd, sd))
    check_parity(host(y), (x.astype(np.float32) @ w32.T).astype(np.float16), plan)
