"""The few-row NF4 product (csrc/nf4_gemm_few.hip), 9 to 64 rows: unsplit and
split, its sums added by the reduce, the norm's launch or another kernel."""

import numpy as np
import pytest
import torch

from oracle import oracle as o
from tests.conftest import beyond_rounding_error
from tests.gpuutil import bits, dt_code, from_bits, randn_bits
from tests.nf4data import oracle_args, random_layer, to_linear


@pytest.fixture(scope="module")
def nf4():
    from ttspipe_amd import fusedops, nf4gemv

    assert nf4gemv.install() and fusedops.install()
    return nf4gemv


def _splits(M, K, rows):
    from ttspipe_amd import _lib

    return _lib.load().ttsp_nf4_gemm_few_splits(M, K, rows)


def test_few_row_split_plan():
    """9 to 64 rows; the most splits up to 4 that fit one workgroup to a CU and
    leave each of a workgroup's four waves two K-steps."""
    for M, K in ((9728, 2560), (6144, 2560), (2560, 9728), (2560, 4096), (1536, 1024), (30, 128), (1000, 512)):
        assert _splits(M, K, 8) == _splits(M, K, 65) == 0
        for rows in (9, 16, 17, 32, 33, 64):
            sp, tiles = _splits(M, K, rows), -(-M // 32)
            assert sp in (1, 2, 4)
            assert sp == 1 or (tiles * sp <= 256 and K // 64 // (4 * sp) >= 2)
            assert sp == 4 or tiles * sp * 2 > 256 or K // 64 // (8 * sp) < 2
    assert _splits(1 << 20, 1 << 14, 16) == 0  # byte offsets past 2^31


def test_long_rows_are_split_at_17_to_32_rows():
    """Past 10240 codes a product of 17 to 32 rows takes the plan's K splits
    (and w1 / w3 two launches, which then split), up to there none."""
    from ttspipe_amd import _lib

    lib = _lib.load()
    for M in (256, 1024, 2560):
        for rows in (17, 24, 32):
            for K in (2560, 9728, 10240):
                assert lib.ttsp_nf4_gemm_splits(M, K, rows) == 1
                assert lib.ttsp_nf4_gemm_swiglu_fits(M, K, rows, 64, 256, 1) == 1
            for K in (10368, 16384, 40960):
                sp = lib.ttsp_nf4_gemm_splits(M, K, rows)
                assert sp == lib.ttsp_nf4_gemm_tile_splits(M, K, rows) and K % (128 * sp) == 0
                assert sp > 1 or K % 256  # (10368 = 81 x 128: no even split)
                assert lib.ttsp_nf4_gemm_swiglu_fits(M, K, rows, 64, 256, 1) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("shape,rows,nested,bs,bs2,dtype", [
    ((9728, 2560), 9, True, 64, 256, torch.bfloat16),     # the fewest rows: 7 of 16 loaded rows repeat
    ((6144, 2560), 16, False, 64, 0, torch.float16),
    ((9730, 2560), 17, True, 128, 256, torch.bfloat16),   # M % 4 == 2, 128-code blocks
    ((2560, 9728), 32, True, 64, 16, torch.float16),      # long runs: scales resolved three times; small groups
    ((2560, 9728), 33, True, 64, 256, torch.bfloat16),    # two column blocks, one with one row
    ((1022, 4096), 64, False, 256, 0, torch.float16),     # a split with M % 4 == 2
    ((33, 128), 24, True, 64, 256, torch.bfloat16),       # two K-steps for four waves; a tile with one row
    ((64, 384), 40, True, 128, 32, torch.float16),        # six K-steps over four waves
    ((96, 16384), 20, True, 64, 256, torch.bfloat16),     # eight splits by the plan
    ((96, 10240), 32, True, 64, 256, torch.float16),      # the longest unsplit row: 40 steps a wave
    ((70, 24576), 17, False, 128, 0, torch.bfloat16),     # eight splits, M % 4 == 2
    ((64, 10368), 31, True, 64, 256, torch.bfloat16),     # past it, no even split: unsplit
])
def test_few_rows_against_fp64(nf4, orc, shape, rows, nested, bs, bs2, dtype):
    """`matmul` and, where it splits, `matmul_partials` and `matmul_norm`:
    the products within the 2e-3 bar beyond rounding; nothing stored past N."""
    (M, K), dt = shape, dt_code(dtype)
    layer = random_layer(M, K, nested, seed=M + rows, bs=bs, bs2=bs2 or 256)
    lin = to_linear(layer, dtype)
    assert nf4.prepare(lin)
    xb = randn_bits(rows * K, dtype, seed=rows, scale=0.5)
    x = from_bits(xb, dtype).view(rows, K)
    ref = orc.nf4_gemm_ref(xb.reshape(rows, K), dt, **oracle_args(layer), M=M, K=K, N=rows, bs=bs,
                           bs2=bs2 or 256).astype(np.float64).reshape(rows, M)
    guard = torch.full((rows + 1, M), 7.0, dtype=dtype, device="cuda")
    nf4.matmul(lin, x, out=guard[:rows])
    assert bool((guard[rows] == 7.0).all())
    assert beyond_rounding_error(o.to_f32(bits(guard[:rows]), dt).reshape(rows, M), ref, dt) < 2e-3
    part = nf4.matmul_partials(lin, x, span=True)
    assert (part is None) == (_splits(M, K, rows) == 1)
    if part is not None:
        work, sp = part
        assert sp == _splits(M, K, rows)
        y = work.double().sum(0).to(dtype)
        assert beyond_rounding_error(o.to_f32(bits(y), dt).reshape(rows, M), ref, dt) < 2e-3


@pytest.mark.gpu
@pytest.mark.parametrize("shape,rows,epi,nested,dtype", [((2560, 9728), 24, 1, True, torch.bfloat16),
                                                         ((2560, 4096), 9, 1, False, torch.float16),
                                                         ((1536, 2048), 32, 0, True, torch.bfloat16),
                                                         ((4088, 2048), 17, 2, True, torch.float16),
                                                         ((2560, 9728), 50, 1, True, torch.bfloat16)])
def test_few_row_norm_equals_its_sums_reduced_then_normed(nf4, shape, rows, epi, nested, dtype):
    """`matmul_norm(span=True)`: its first output is the sums of
    `matmul_partials` added in split order with the epilogue's roundings, its
    second `fusedops.rms_norm` of it, bit for bit."""
    from ttspipe_amd import fusedops

    M, K = shape
    lin = to_linear(random_layer(M, K, nested, seed=M + rows), dtype)
    assert nf4.prepare(lin)
    x = from_bits(randn_bits(rows * K, dtype, seed=rows, scale=0.5), dtype).view(1, rows, K)
    r = from_bits(randn_bits(rows * M, dtype, seed=rows + 1), dtype).view(1, rows, M) if epi else None
    g = torch.rand(M, generator=torch.Generator().manual_seed(M)).add(0.5).to(dtype).cuda()
    y, yn = nf4.matmul_norm(lin, x, g, 1e-5, epi=epi, operand=r, span=True)
    work, sp = nf4.matmul_partials(lin, x, span=True)
    acc = work[0].clone()
    for z in range(1, sp):
        acc += work[z]
    expect = acc.to(dtype).view(1, rows, M)
    if epi == 1:
        expect = r + expect
    if epi < 2:  # (the gate's exp is the kernels' own)
        assert torch.equal(y.view(torch.int16), expect.view(torch.int16))
    else:
        silu = torch.nn.functional.silu(r.double()).to(dtype)
        assert ((y.double() - (silu * expect).double()).norm() / y.double().norm()).item() < 4e-3
    assert torch.equal(yn.view(torch.int16), fusedops.rms_norm(y, g, 1e-5).view(torch.int16))
