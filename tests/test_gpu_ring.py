"""GPU parity of the few-tile GEMM (ring_gemm_kernel): calls of 33 rows and more whose grid is
small, and some of fewer rows, take it without a flag, with 16, 32 or 64 rows per workgroup, over the whole K or in slices.

Bars as for every linear (rel-L2 <= 1e-3 against the oracle, the reference's rounding-budget gate); identity
inputs with power-of-two scales are bit-exact; two calls agree bit for bit.
"""
import numpy as np
import pytest
import torch

import lowbit_hip
from conftest import announce
from oracle import lowbit_oracle as o
from test_gpu_linear import check, problem, run, to_dev

pytestmark = pytest.mark.gpu

# (fmt, M, N, K, group, rank, bias): the last stage's 32 / 64 / 96 codes and whole stages, K below a stage and
# around the ring's depth, rows and columns at the edges of the 16 / 32 / 64-row tiles, scales of 8 and 28 KB,
# corrections of one to four eights
CASES = [
    ('int4', 33, 64, 32, 32, 0, False), ('int4', 48, 65, 64, 64, 0, True), ('int4', 40, 63, 96, 32, 0, False),
    ('int4', 37, 200, 128, 128, 0, False), ('int4', 64, 129, 160, 32, 0, True), ('nf4', 50, 192, 576, 32, 0, False),
    ('nf4', 333, 2560, 960, 64, 0, True), ('nf4', 97, 1000, 992, 32, 0, False), ('nf4', 17, 40, 640, 64, 0, False),
    ('int8', 31, 33, 768, 768, 0, True), ('int8', 100, 700, 896, 64, 0, False), ('int8', 256, 576, 576, 576, 32, False),
    ('int8', 256, 1536, 576, 576, 32, True), ('int8', 257, 1500, 1504, 1504, 8, False), ('int4', 65, 190, 1056, 32, 24, True),
    ('nf4', 129, 577, 224, 32, 16, False), ('int4', 48, 14336, 1024, 128, 0, False), ('int4', 500, 320, 2080, 32, 0, True),
    ('int4', 64, 500, 4096, 32, 0, False), ('int4', 600, 2048, 2048, 2048, 0, False), ('int8', 513, 2040, 2048, 2048, 0, True),
    # up to 32 rows: short rows, many columns, large weights, and every row count class of a correction
    ('int8', 17, 1536, 576, 576, 0, True), ('int8', 32, 4100, 2304, 2304, 0, False), ('int4', 31, 576, 1536, 64, 0, False),
    ('int4', 20, 4160, 2560, 32, 0, True), ('nf4', 20, 8190, 256, 128, 0, False), ('int4', 9, 11072, 4096, 128, 0, False),
    ('int8', 2, 100, 96, 96, 8, True), ('int8', 16, 577, 640, 640, 32, False), ('int8', 19, 64, 4096, 4096, 16, False),
    ('int4', 5, 130, 320, 64, 24, True), ('nf4', 32, 70, 96, 32, 32, False),
    # past one round of 64-row tiles, where the kernel is estimated the faster one and where not; 17 rows over two rounds
    ('int4', 1000, 2000, 2048, 64, 0, True), ('int8', 50, 16500, 2080, 2080, 0, False), ('int8', 320, 4900, 2048, 2048, 0, True),
    ('int4', 320, 6912, 2048, 64, 0, False), ('int8', 17, 17000, 2048, 2048, 0, True),
    # both sides of the lines of short rows, of pairs of tiles, of groups of 32 and of 9 to 16 rows
    ('int4', 340, 2740, 512, 64, 0, False), ('int4', 340, 2740, 544, 32, 0, True), ('nf4', 321, 2750, 384, 64, 0, True),
    ('int4', 19, 7588, 640, 128, 0, False), ('int4', 19, 7000, 704, 64, 0, True), ('nf4', 70, 90, 3072, 32, 0, True),
    ('nf4', 20, 8300, 640, 64, 0, False), ('nf4', 20, 8300, 672, 32, 0, True), ('int8', 9, 17000, 2816, 2816, 0, False),
]


@pytest.mark.parametrize('spec', CASES, ids=lambda s: '-'.join(map(str, s)))
def test_ring_matches_oracle(device, spec):
    fmt, m, n, k, group, rank, bias = spec
    announce('ring', spec)
    p = problem(np.random.default_rng(m * 977 + n + k + group), fmt, m, n, k, group, rank=rank, bias=bias)
    got = run(p, device)
    check(p, got, f'ring {spec}')
    assert np.array_equal(run(p, device), got)


def test_ring_fp16_rows(device):
    """fp16 weights (no scales) against a double product, a ragged last stage included."""
    announce('ring fp16')
    rng = np.random.default_rng(3)
    for m, n, k in ((40, 70, 96), (256, 576, 576), (65, 300, 1536), (100, 2050, 4128), (330, 2700, 3104), (330, 2700, 544), (50, 1000, 6400)):
        x = rng.standard_normal((m, k)).astype(np.float16)
        w = (rng.standard_normal((n, k)) * 0.02).astype(np.float16)
        y = lowbit_hip.linear(to_dev(x, device), to_dev(w, device), None, format='fp16', N=n, K=k, group_size=k)
        assert o.rel_l2(y.cpu().numpy(), x.astype(np.float64) @ w.astype(np.float64).T) <= 1e-3, (m, n, k)


@pytest.mark.parametrize('m,n', [(64, 128), (250, 1000)])
def test_ring_identity_is_bit_exact(device, m, n):
    k, group = 480, 32
    announce('ring identity', m, n)
    rng = np.random.default_rng(16)
    data = o.pack(rng.integers(0, 16, n * k).astype(np.uint8))
    scales = (2.0 ** rng.integers(-10, 3, n * (k // group))).astype(np.float16)
    w = o.dequantize('int4', (n, k), group, data, scales.tobytes())
    x = np.zeros((m, k), np.float16)
    cols = rng.integers(0, k, m)
    x[np.arange(m), cols] = 1.0
    y = lowbit_hip.linear(to_dev(x, device), to_dev(np.frombuffer(data, np.uint8), device), to_dev(scales, device),
                          format='int4', N=n, K=k, group_size=group).cpu().numpy()
    np.testing.assert_array_equal(y, w[:, cols].T)


@pytest.mark.parametrize('columns,pitch', [(200, 208), (203, 211)])
def test_ring_strided_rows_leave_the_rest(device, columns, pitch):
    """Strided x and y (16-byte rows and odd ones): the columns past N keep their values; a row of infinities
    and a NaN stay in their rows."""
    announce('ring strided', columns, pitch)
    m, k = 70, 352
    p = problem(np.random.default_rng(5), 'int4', m, columns, k, 32)
    wide = torch.full((m, k + 16), float('nan'), dtype=torch.float16, device=device)
    wide[:, :k] = to_dev(p['x'], device)
    wide[3, 5], wide[9, 351] = float('inf'), float('nan')
    y = torch.full((m, pitch), 7.0, dtype=torch.float16, device=device)
    lowbit_hip.linear(wide[:, :k], to_dev(np.frombuffer(p['data'], np.uint8), device),
                      to_dev(np.frombuffer(p['scales'], np.float16), device), format='int4', N=columns, K=k,
                      group_size=32, out=y[:, :columns])
    got = y.cpu().numpy()
    assert (got[:, columns:] == 7.0).all()
    assert not np.isfinite(got[3, :columns]).all() and np.isnan(got[9, :columns]).all()
    rows = [r for r in range(m) if r not in (3, 9)]
    check(dict(p, x=p['x'][rows], m=len(rows)), got[rows][:, :columns], 'ring strided')


# (fmt, M, N, K, group, bias): K slices of whole and ragged ends (the last stage of 32 and 96 codes, a last slice
# shorter than the others), both row tiles, plans of tile_rows / wide_rows / the split GEMM, the lines of the rule, and
# rows that wide_rows_kernel does not cut (11008 codes of int8)
SLICED = [('int8', 17, 1000, 3104, 3104, True), ('int8', 32, 4096, 4096, 4096, False), ('int4', 24, 200, 4160, 64, True),
          ('nf4', 33, 130, 3168, 3168, False), ('int4', 64, 577, 8192, 128, True), ('int8', 100, 65, 8224, 8224, False),
          ('nf4', 129, 192, 4096, 64, True), ('int4', 20, 2048, 8192, 128, False), ('nf4', 32, 4096, 4096, 128, True),
          ('int8', 19, 512, 11008, 11008, True), ('int4', 17, 320, 14336, 14336, False),
          # 16-row tiles: 9 to 16 rows, and 5 to 8 of NF4 and INT8
          ('int4', 9, 3072, 8192, 128, True), ('int8', 16, 3137, 8224, 8224, False), ('nf4', 5, 4109, 11008, 64, True),
          ('int8', 8, 3200, 14336, 14336, True)]


@pytest.mark.parametrize('spec', SLICED, ids=lambda s: '-'.join(map(str, s)))
def test_ring_slices_match_oracle(device, spec):
    """The oracle, bit-equal repeats, and rows of infinities and NaN that stay in their rows."""
    fmt, m, n, k, group, bias = spec
    announce('ring slices', spec)
    p = problem(np.random.default_rng(m + n + k), fmt, m, n, k, group, rank=0, bias=bias)
    got = run(p, device)
    check(p, got, f'ring slices {spec}')
    assert np.array_equal(run(p, device), got)
    x = p['x'].copy()
    x[1, k - 1], x[m - 1, 3] = np.inf, np.nan
    bad = run(dict(p, x=x), device)
    rows = [r for r in range(m) if r not in (1, m - 1)]
    assert np.array_equal(bad[rows], got[rows]) and np.isnan(bad[m - 1]).all() and not np.isfinite(bad[1]).any()
