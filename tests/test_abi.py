"""The C-ABI library loads, exports every symbol the header declares, and
rejects malformed requests before any GPU work (CPU-only checks)."""
import ctypes
import re
from pathlib import Path

import pytest

from ondeviceinfer_amd import _native

HEADERS = sorted((Path(__file__).resolve().parents[1] / 'include').glob('*.h'))


def declared_functions() -> list[str]:
    names = []
    for header in HEADERS:
        text = re.sub(r'/\*.*?\*/', '', header.read_text(), flags=re.S)
        names += re.findall(r'^\s*(?:const\s+char\s*\*|int)\s+(wq_\w+)\s*\(', text, flags=re.M)
    return names


def test_header_declares_the_bound_entry_points():
    names = declared_functions()
    assert len(names) == len(set(names)) >= 12
    assert set(names) == set(_native.EXPORTED_SYMBOLS)


def test_library_exports_every_declared_symbol():
    lib = _native.load()
    for name in declared_functions():
        assert hasattr(lib, name), name
    assert lib.wq_abi_version() == _native.ABI_VERSION


def _status(fn, *args):
    return getattr(_native.load(), fn)(*args)


def test_shape_validation_happens_on_the_host():
    tb, mb = ctypes.c_size_t(), ctypes.c_size_t()
    assert _status('wq_w4_repack_size', 5120, 5120, 128, ctypes.byref(tb), ctypes.byref(mb)) == _native.WQ_OK
    assert tb.value == 5120 * 5120 // 2 and mb.value == 320 * 40 * 40
    assert _status('wq_w4_repack_size', 12, 5120, 128, ctypes.byref(tb), ctypes.byref(mb)) == _native.WQ_ERR_UNSUPPORTED
    assert b'n % 8' in _native.load().wq_last_error()
    assert _status('wq_w4_repack_size', 16, 5120, 64, ctypes.byref(tb), ctypes.byref(mb)) == _native.WQ_ERR_UNSUPPORTED
    assert _status('wq_w4_repack_size', 0, 5120, 128, ctypes.byref(tb), ctypes.byref(mb)) == \
        _native.WQ_ERR_INVALID_ARGUMENT
    # k not a multiple of the group -> rejected before any launch
    assert _status('wq_w4a16_linear', 1, 1, 200, 1, 1, 16, 128, 1, None, 0, None) == _native.WQ_ERR_UNSUPPORTED
    # null pointers -> rejected
    assert _status('wq_w4a16_linear', None, 1, 256, None, None, 16, 128, None, None, 0, None) == \
        _native.WQ_ERR_INVALID_ARGUMENT
    assert _status('wq_w8_quantize', None, 0, 4, None, None, None, None) == _native.WQ_ERR_INVALID_ARGUMENT


def test_status_maps_to_python_exceptions():
    with pytest.raises(ValueError, match='n % 8'):
        _native.w4_repack_size(12, 256, 128)
    assert _native.w4_repack_size(16, 256, 128) == (16 * 128, 2 * 40)
    assert _native.w4a16_workspace_size(1, 5120, 5120, 128) == 0


def test_prefill_k_split_workspace_follows_the_chain_length():
    """The deep-ring GEMM's k split, as the host sizes its workspace (no GPU
    needed): a 16 KiB counter region plus one fp32 partial tile set of
    4 waves x NT x MT KiB per (workgroup, split), NT = 1 and MT = 2 (32-row
    tiles) at these M.  Short chains (40 blocks) split only grids of at
    most 384 workgroups, long ones (64 blocks or more) up to 640."""
    counters, per_split_tile = 16384, 4 * 1 * 2 * 1024
    # down 17408->5120 (136 blocks): 80 n slices x 4 / 8 row blocks
    assert _native.w4a16_workspace_size(128, 5120, 17408, 128) == counters + 320 * 4 * per_split_tile
    assert _native.w4a16_workspace_size(256, 5120, 17408, 128) == counters + 640 * 2 * per_split_tile
    # q/o 5120->5120 (40 blocks) at M = 256: 640 workgroups keep the whole k range
    assert _native.w4a16_workspace_size(256, 5120, 5120, 128) == 0
    # fused QKV 5120->7168 (40 blocks): 112 n slices x 3 row blocks at M = 65 split
    # in four; 4 row blocks at M = 128 (448 workgroups) keep the whole k range
    assert _native.w4a16_workspace_size(65, 7168, 5120, 128) == counters + 336 * 4 * per_split_tile
    assert _native.w4a16_workspace_size(128, 7168, 5120, 128) == 0
    assert _native.w4a16_workspace_size(256, 5120, 5120, 128) == 0
    # 65 blocks, 16 n slices x 22 row blocks = 352 workgroups: four splits
    assert _native.w4a16_workspace_size(700, 1000, 8320, 128) == counters + 352 * 4 * per_split_tile
    # M = 257: 64-row tiles (400 workgroups), no deep ring, no split
    assert _native.w4a16_workspace_size(257, 5120, 17408, 128) == 0


def test_the_library_says_which_workspaces_start_zeroed():
    """The bytes a caller zero-fills come from the library's own plan (no GPU
    needed): the counter region where a kernel counts arrivals, else none, and
    no copy of that rule in the Python binding."""
    counters = 16384
    for m, n, k, zeroed in ((1, 5120, 17408, counters),     # decode GEMV, k split
                            (1, 5120, 5120, 0),             # decode GEMV, whole k: no workspace
                            (24, 7168, 5120, counters),     # short chains of 12 to 32 rows: the last arriver sums
                            (40, 7168, 5120, 0),            # a second launch sums
                            (56, 5120, 17408, 0),
                            (128, 5120, 17408, counters),   # deep-ring GEMM, k split
                            (4096, 5120, 5120, 0)):
        assert _native.w4a16_workspace_zeroed(m, n, k, 128) == zeroed, (m, n, k)
        assert zeroed <= _native.w4a16_workspace_size(m, n, k, 128)
    assert not hasattr(_native, '_counts_arrivals')
    assert _status('wq_w4a16_workspace_zeroed', 1, 0, 128, 128, None) == _native.WQ_ERR_INVALID_ARGUMENT


def test_w8a8_256_tiles_stop_where_their_reads_leave_the_buffer_range():
    """256 rows of k bytes end at 2^31 for k = 2^23, one byte past the 31-bit
    record count of a buffer (the last reads would come back as zeros): that k
    takes the 128-row tiles, one 128-k block less the 256 x 256 ones."""
    m = n = 3584
    assert _native.linear_plan('w8a8', m, n, (1 << 23) - 128) == 'gemm 256x256'
    assert _native.linear_plan('w8a8', m, n, 1 << 23) == 'gemm 2x8'
    assert _native.linear_plan('w8a8', m, n, (1 << 23) + 128) == 'gemv'
    assert _native.linear_plan('w8a8', 2048, 7168, 5120) == 'gemm 256x256'
    with pytest.raises(ValueError):
        _native.linear_plan('w8a8', 2048, 7168, 5100)


def test_w4_rows_5_to_64_take_the_kernel_estimated_faster():
    """Short narrow chains stay on the skinny kernels at every row count (the
    shared-activation kernel takes 1.3 to 2 times as long there), long or wide
    ones leave them, and no row count between two others makes an exception."""
    plan = lambda m, n, k: _native.linear_plan('w4a16', m, n, k).split()[0]
    rows = range(5, 65)
    for n, k in ((512, 512), (2048, 1024), (6144, 512), (1024, 1024), (4040, 1024)):
        assert {plan(m, n, k) for m in rows} == {'skinny'}, (n, k)
    for n, k in ((5120, 17408), (17408, 5120), (12288, 12288), (1024, 12288)):
        assert {plan(m, n, k) for m in rows} == {'mid'}, (n, k)
    for n, k in ((1024, 5120), (5120, 5120), (7168, 5120), (6144, 2048), (12288, 2048)):
        taken = [plan(m, n, k) == 'mid' for m in rows if not 12 <= m <= 32]   # 12..32: other partial sums
        assert taken == sorted(taken), (n, k)
    assert {plan(m, 17408, 1024) for m in range(12, 33)} == {plan(m, 12288, 2048) for m in range(12, 33)} == {'batch'}
    for m in (33, 34, 35):
        for n, k in ((1024, 5120), (5120, 5120), (7168, 5120), (17408, 5120), (12288, 2048)):
            assert plan(m, n, k) == 'mid', (m, n, k)
    assert plan(33, 34816, 1024) == 'deep' and plan(33, 34816, 5120) == 'mid'


def test_int8_rows_5_to_64_take_the_kernel_estimated_faster():
    plan = lambda m, n, k: _native.linear_plan('w8a16', m, n, k).split()[0]
    rows = range(5, 65)
    for n, k in ((512, 512), (2048, 512), (6144, 512), (4040, 512)):
        assert {plan(m, n, k) for m in rows} == {'skinny'}, (n, k)
    for n, k in ((5120, 17408), (17408, 5120), (34816, 5120), (9216, 12288)):
        assert {plan(m, n, k) for m in rows} == {'mid'}, (n, k)
    for n, k in ((1024, 5120), (5120, 5120), (6144, 1024), (4040, 5120), (17408, 2048)):
        taken = [plan(m, n, k) == 'mid' for m in rows]
        assert taken == sorted(taken), (n, k)
    assert plan(8, 1024, 5120) == plan(33, 2048, 512) == 'skinny' and plan(24, 1024, 5120) == 'mid'


def test_w8a8_rows_5_to_255_take_the_kernel_estimated_faster():
    plan = lambda m, n, k: _native.linear_plan('w8a8', m, n, k).split()[0]
    for n, k in ((512, 512), (1024, 2048), (4040, 2048), (9216, 512)):
        assert 'mid' not in {plan(m, n, k) for m in range(5, 201)}, (n, k)
    for n, k in ((1024, 17408), (5120, 17408), (7168, 8192)):
        assert {plan(m, n, k) for m in range(17, 129)} == {'mid'}, (n, k)
    assert {plan(m, 34816, 5120) for m in range(5, 65)} == {'mid'} and plan(129, 34816, 5120) == 'gemm'
    assert plan(8, 5120, 5120) == 'gemv' and plan(16, 5120, 5120) == plan(48, 17408, 5120) == 'mid'
    assert plan(200, 13000, 3328) == 'mid' and plan(96, 13000, 3328) == plan(200, 17408, 5120) == 'gemm'


def test_every_prefill_grid_is_reached_and_tested():
    """The GPU test's shapes run the grids it names, cover the cost table's
    nine plain grids, and have each fused epilogue on every grid it exists on."""
    from test_gpu_gemm_grids import EVERY_GRID
    assert list(EVERY_GRID) == ['1x4', '2x4', '2x5', '2x6', '2x8', '4x4', '4x6', '4x7', '4x8']
    for grid, shapes in EVERY_GRID.items():
        for fmt in ('w4a16', 'w8a16'):
            for shape in shapes:
                assert _native.linear_plan(fmt, *shape) == f'gemm {grid}', (fmt, shape)
            modes = {e for e in (_native.EPI_SILU_MUL, _native.EPI_RESIDUAL) for m, n, k in shapes
                     if (_native.w4a16_epilogue_supported(m, n, k, 128, e) if fmt == 'w4a16'
                         else _native.w8a16_epilogue_supported(m, n, k, e))
                     and _native.linear_plan(fmt, m, n, k, e) == f'gemm {grid}'}
            assert modes == ({2} if grid == '1x4' else {1, 2}), (fmt, grid, modes)
    # Costs follow the whole round: narrow tiles on short chains, the wide ones' lead on long ones.
    assert _native.linear_plan('w8a16', 128, 34816, 5120) == 'gemm 2x4'
    assert _native.linear_plan('w4a16', 4096, 17408, 5120) == _native.linear_plan('w8a16', 4096, 34816, 5120) == 'gemm 4x8'
    assert _native.linear_plan('w4a16', 65, 5120, 1280) == 'deep 1x2x1'
