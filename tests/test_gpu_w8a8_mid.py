"""W8A8 at 5 to 255 rows (the shared-activation kernel with its k splits) and
the quantizer's register-resident rows, bit for bit against the oracle."""
import numpy as np
import pytest
import torch

from oracle import qdq
from ondeviceinfer_amd import _native

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to('cuda:0')


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


# Both ends of the 16-row chunks and of the row blocks.  k = 8320 (65 blocks, a
# long chain with a ragged last stage: splits), 2688 (21 blocks) and 2944 (23);
# n: a partial last tile group, groups of ten tiles (16400: two splits; 33000
# one), and 13000 x 128: the shapes below the size that stay on the GEMM.
@pytest.mark.parametrize('n,k,ms', [(512, 2688, (17, 64)), (4104, 2688, (17, 33, 48, 49, 97)),
                                    (1001, 8320, (5, 16, 17, 33, 64, 96, 128, 129, 255)),
                                    (7168, 2944, (9, 32, 49, 65, 128, 129, 200)), (16400, 1280, (5, 17, 48, 64, 65, 128)),
                                    (33000, 640, (5, 64, 65, 200)), (13000, 128, (9, 40))])
def test_w8a8_mid_bit_exact_in_both_layouts(n, k, ms):
    rng = np.random.default_rng(n + k)
    m = max(ms)
    qx = rng.integers(-127, 128, (m, k)).astype(np.int8)
    qw = rng.integers(-127, 128, (n, k)).astype(np.int8)
    xs = (rng.random(m) * 0.05 + 1e-4).astype(np.float32)
    wsc = (rng.random(n) * 0.002 + 1e-5).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float16)
    expected = qdq.w8a8_linear_int(qx, xs, qw, wsc, bias).view(np.uint16)
    row_major, args = dev(qw), (dev(wsc), dev(bias))
    tiles = _native.w8_repack(row_major)
    lib = _native.load()
    for rows in ms:
        print(f'[w8a8 mid] m={rows} n={n} k={k}', flush=True)
        xd, sd = dev(qx[:rows]), dev(xs[:rows])
        for w in (row_major, tiles):
            got = host(_native.w8a8_linear(xd, sd, w, *args)).view(np.uint16)
            assert np.array_equal(got, expected[:rows])
        # the entry point without a workspace: the unsplit kernels, the same bits
        y = torch.empty(rows, n, dtype=torch.float16, device='cuda:0')
        assert lib.wq_w8a8_linear(xd.data_ptr(), sd.data_ptr(), rows, k, row_major.data_ptr(), args[0].data_ptr(), n,
                                  args[1].data_ptr(), y.data_ptr(), torch.cuda.current_stream().cuda_stream) == 0
        assert np.array_equal(host(y).view(np.uint16), expected[:rows])


# Shapes the kernel takes: one to eight 16-row chunks, two row blocks, splits, ten-tile groups unsplit and in two
# splits, partial last tile groups and stages.
@pytest.mark.parametrize('m,n,k', [(17, 1001, 8320), (64, 1001, 8320), (96, 1001, 8320), (128, 1001, 8320),
                                   (255, 1001, 8320), (16, 7176, 5248), (33, 7176, 5248), (192, 7176, 5248),
                                   (5, 33000, 4224), (49, 17400, 5120), (128, 17400, 5120)])
def test_w8a8_mid_shapes_bit_exact(m, n, k):
    plan = _native.linear_plan('w8a8', m, n, k)
    print(f'[w8a8 mid] m={m} n={n} k={k}: {plan}', flush=True)
    assert plan.startswith('mid')
    rng = np.random.default_rng(n + k + m)
    qx, qw = (rng.integers(-127, 128, s, dtype=np.int8) for s in ((m, k), (n, k)))
    xs, wsc = ((rng.random(s) * 0.01 + 1e-4).astype(np.float32) for s in (m, n))
    tiles = _native.w8_repack(dev(qw))
    got = host(_native.w8a8_linear(dev(qx), dev(xs), tiles, dev(wsc)))
    lib, y = _native.load(), torch.empty(m, n, dtype=torch.float16, device='cuda:0')
    td = (dev(qx), dev(xs), dev(wsc))
    assert lib.wq_w8a8_linear_tiled(td[0].data_ptr(), td[1].data_ptr(), m, k, tiles.tiles.data_ptr(), td[2].data_ptr(),
                                    n, None, y.data_ptr(), torch.cuda.current_stream().cuda_stream) == 0
    assert np.array_equal(got.view(np.uint16), host(y).view(np.uint16))   # without the splits' workspace
    rows, cols = sorted({0, 15, m // 2, m - 1} & set(range(m))), np.r_[0:32, n // 2:n // 2 + 16, n - 40:n]
    expected = qdq.w8a8_linear_int(qx[rows], xs[rows], qw[cols], wsc[cols], None)
    assert np.array_equal(got[rows][:, cols].view(np.uint16), expected.view(np.uint16))


# 1024 threads a row (m <= 512) with one and three chunks a thread, 256 threads with
# one, three and nine, and rows too long to stay in registers.
@pytest.mark.parametrize('m,k', [(7, 2056), (48, 8192), (512, 8200), (2, 24576), (513, 2048), (600, 5120), (530, 17408),
                                 (3, 40000)])
def test_w8a8_quantize_register_rows_bit_exact(m, k):
    rng = np.random.default_rng(m + k)
    x = (rng.standard_normal((m, k)) * np.exp(rng.uniform(-9, 6, (m, 1)))).astype(np.float16)
    x[0] = np.float16(6e-8) * rng.integers(-3, 4, k)       # subnormal values
    x[-1, ::3] = np.float16(65504)
    qx, sx = _native.w8a8_quantize(dev(x))
    q_ref, s_ref = qdq.quantize_activations_per_token(x)
    assert np.array_equal(host(qx), q_ref) and np.array_equal(host(sx), s_ref)


def test_w8a8_quantize_non_finite_rows():
    """An infinite value makes its row's scale infinite: finite values give 0
    (v / inf), the infinite ones and NaN the clamp of NaN, -127; a NaN alone
    leaves the scale to the other values."""
    x = np.ones((3, 5120), dtype=np.float16)
    x[0, 7], x[0, 9], x[1, 5] = np.inf, -np.inf, np.nan
    qx, sx = (host(t) for t in _native.w8a8_quantize(dev(x)))
    assert np.isinf(sx[0]) and sx[1] == sx[2] == np.float32(1) / np.float32(127)
    row = np.zeros(5120, dtype=np.int8)
    row[[7, 9]] = -127
    assert np.array_equal(qx[0], row)
    row = np.full(5120, 127, dtype=np.int8)
    assert np.array_equal(qx[2], row)
    row[5] = -127
    assert np.array_equal(qx[1], row)


@pytest.mark.parametrize('m,n,k,bias', [(4000, 4040, 256, False), (3900, 4088, 128, True), (2000, 8190, 384, True),
                                        (2048, 7168, 640, False)])
def test_w8a8_256_tiles_exact(gpu, m, n, k, bias):
    """256 x 256 tiles (long batches over INT8 tiles; ragged rows and columns, one to five blocks): sampled rows equal
    the integer oracle and every row the row-major GEMM, bit for bit (exact integer sums, one scaling order)."""
    rng = np.random.default_rng(m + n + k)
    qx, qw = (rng.integers(-127, 128, s, dtype=np.int8) for s in ((m, k), (n, k)))
    sx, sw = (rng.uniform(1e-3, 1e-2, s).astype(np.float32) for s in (m, n))
    b = rng.standard_normal(n).astype(np.float16) if bias else None
    td = [None if v is None else torch.from_numpy(v).to(gpu) for v in (qx, sx, qw, sw, b)]
    y = _native.w8a8_linear(td[0], td[1], _native.w8_repack(td[2]), td[3], td[4])
    assert torch.equal(y, _native.w8a8_linear(*td))
    rows = [0, 1, 127, 128, 255, 256, m - 17, m - 1]
    acc = qx[rows].astype(np.int64) @ qw.astype(np.int64).T
    want = acc.astype(np.float32) * sx[rows][:, None] * sw[None]
    if bias:
        want = want + b.astype(np.float32)
    assert np.array_equal(y.cpu().numpy()[rows], want.astype(np.float16))
