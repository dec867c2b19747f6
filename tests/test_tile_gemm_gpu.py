"""The tiled NF4 product (csrc/nf4_gemm_tile.hip) in each of its forms: 64, 128
and 256 weight rows a workgroup, one or both K halves, unsplit and split."""

import numpy as np
import pytest
import torch

from oracle import oracle as o
from tests.conftest import beyond_rounding_error
from tests.gpuutil import bits, dt_code, from_bits, randn_bits, split_product
from tests.nf4data import oracle_args, random_layer, to_linear


@pytest.fixture(scope="module")
def nf4():
    from ttspipe_amd import nf4gemv

    assert nf4gemv.install()
    return nf4gemv


def test_tile_splits_follow_the_split_plan():
    """The split plan's, or from 256 rows 1 in place of 2 where the row is too
    wide for the norm's reduce and 2 in place of 4 at 64 to 127 K-steps."""
    from ttspipe_amd import _lib

    lib = _lib.load()
    for M, K in ((9728, 2560), (6144, 2560), (2560, 9728), (2560, 4096), (4096, 2560), (1536, 1024), (1540, 2560)):
        for N in (65, 100, 128, 200, 256, 257, 384, 400, 512):
            plan, tile = lib.ttsp_nf4_gemm_splits(M, K, N), lib.ttsp_nf4_gemm_tile_splits(M, K, N)
            assert tile == plan or (N >= 256 and ((tile == 1 and plan == 2 and M > 4096)
                                                  or (tile == 2 and plan == 4 and 64 <= K // 64 < 128)))


@pytest.mark.gpu
@pytest.mark.parametrize("shape,rows,nested,bs,bs2,dtype,epi", [
    ((64, 128), 65, True, 64, 256, torch.bfloat16, 0),       # KG 2: one K-step a half
    ((70, 384), 129, False, 128, 0, torch.float16, 1),       # three steps a half, one activation row in the last tile
    ((1542, 2688), 200, True, 64, 16, torch.bfloat16, 2),    # 21 steps a half: scales resolved twice; M % 4 == 2
    ((9728, 2560), 256, True, 64, 256, torch.float16, 0),    # 128 rows a workgroup
    ((9000, 2560), 250, False, 256, 0, torch.bfloat16, 1),   # the same, ragged both ways
    ((9730, 2560), 500, True, 64, 32, torch.bfloat16, 0),    # 256 rows a workgroup, M % 4 == 2
    ((8190, 2560), 511, True, 64, 256, torch.float16, 2),    # 128 tiles of 256 rows: 256 of 128 rows run instead
    ((8200, 2560), 512, False, 64, 0, torch.bfloat16, 1),    # one tile more: 256 rows a workgroup
    ((9728, 2176), 512, True, 128, 256, torch.float16, 2),   # 34 steps: a ring remainder of one past two chunks
    ((9728, 2048), 400, False, 64, 0, torch.bfloat16, 0),    # 32 steps: a remainder of two
    ((2560, 9728), 512, True, 64, 256, torch.bfloat16, 1),   # four K splits
])
def test_tile_gemm_against_fp64(nf4, orc, shape, rows, nested, bs, bs2, dtype, epi):
    """Within the 2e-3 bar beyond the output's own rounding, nothing stored
    past N, every epilogue."""
    (M, K), dt = shape, dt_code(dtype)
    layer = random_layer(M, K, nested, seed=M + rows, bs=bs, bs2=bs2 or 256)
    lin = to_linear(layer, dtype)
    assert nf4.prepare(lin)
    xb = randn_bits(rows * K, dtype, seed=rows, scale=0.5)
    x = from_bits(xb, dtype).view(rows, K)
    rb = randn_bits(rows * M, dtype, seed=5)
    guard = torch.full((rows + 1, M), 7.0, dtype=dtype, device="cuda")
    y = nf4.matmul(lin, x, epi=epi, operand=from_bits(rb, dtype).view(rows, M) if epi else None, out=guard[:rows])
    assert bool((guard[rows] == 7.0).all())
    sample = np.unique(np.r_[0:rows:17, rows - 1])
    ref = orc.nf4_gemm_ref(xb.reshape(rows, K)[sample], dt, **oracle_args(layer), M=M, K=K, N=sample.size, bs=bs,
                           bs2=bs2 or 256).astype(np.float64).reshape(sample.size, M)
    if epi:
        ref = o.to_f32(o.from_f32(ref.astype(np.float32), dt), dt).astype(np.float64)
        r = o.to_f32(rb, dt).astype(np.float64).reshape(rows, M)[sample]
        silu = o.to_f32(o.from_f32((r / (1 + np.exp(-r))).astype(np.float32), dt), dt).astype(np.float64)
        ref = r + ref if epi == 1 else silu * ref
    got = o.to_f32(bits(y), dt).reshape(rows, M)[sample]
    assert beyond_rounding_error(got, ref, dt) < 2e-3


@pytest.mark.gpu
@pytest.mark.parametrize("M,rows,nested,dtype", [(6144, 385, True, torch.bfloat16), (6144, 400, False, torch.float16),
                                                 (6144, 512, True, torch.bfloat16), (6146, 511, True, torch.float16)])
def test_span_partial_sums_against_fp64(nf4, orc, M, rows, nested, dtype):
    """A prompt block's wqkv: `matmul_partials(span=True)` in the plan's two
    splits of 2560 codes, its sums added in order against the fp64 product,
    ragged M and rows. The bar on the fp32 sums themselves, 1e-5 of the largest:
    160 roundings of 2^-24 in a random walk are 8e-7 of a sum's deviation, 5
    times that over 1e5 of them."""
    from ttspipe_amd import _lib

    K, dt = 2560, dt_code(dtype)
    assert _lib.load().ttsp_nf4_gemm_splits(M, K, rows) == 2
    layer = random_layer(M, K, nested, seed=M + rows)
    lin = to_linear(layer, dtype)
    assert nf4.prepare(lin)
    xb = randn_bits(rows * K, dtype, seed=rows, scale=0.5)
    work, splits = nf4.matmul_partials(lin, from_bits(xb, dtype).view(rows, K), span=True)
    assert splits == 2
    sample = np.unique(np.r_[0:rows:29, rows - 1])
    ref = orc.nf4_gemm_ref(xb.reshape(rows, K)[sample], dt, **oracle_args(layer), M=M, K=K, N=sample.size, bs=64,
                           bs2=256).astype(np.float64).reshape(sample.size, M)
    got = (work[0] + work[1]).cpu().numpy().astype(np.float64)[sample]
    assert np.abs(got - ref).max() < 1e-5 * np.abs(ref).max()


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,rows", [(1024, 1024, 128), (6144, 2560, 385), (6144, 2560, 512), (2560, 4096, 300)])
@pytest.mark.parametrize("epi", [1, 2])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_epilogue_over_all_operands_equals_the_reduce_kernels(nf4, M, K, rows, epi, dtype):
    """The tile kernel's residual and gate, eight values at a time, against the
    split reduce's, one by one, bit for bit: one-hot rows of X make a product
    that no order of sums changes, and the operands run over every finite value
    of the type, both infinities and NaN (which stays a NaN)."""
    from ttspipe_amd import _lib

    lin = to_linear(random_layer(M, K, True, seed=6), dtype)
    assert nf4.prepare(lin)
    x = torch.zeros(rows, K, dtype=dtype, device="cuda")
    x[torch.arange(rows), (torch.arange(rows) * 37) % K] = 1.0
    r = torch.arange(rows * M, device="cuda").to(torch.int16).view(dtype).view(rows, M).contiguous()
    f, lib, out = lin._nf4_fast, _lib.load(), torch.empty(rows, M, dtype=dtype, device="cuda")
    rc = lib.ttsp_nf4_gemm(x.data_ptr(), _lib.dtype_code(dtype), f["w"], f["a8"], f["amax"], f["code2"], f["offset"],
                           f["lut"].data_ptr(), out.data_ptr(), r.data_ptr(), epi, M, K, rows, 64, 256, _lib.stream())
    splits = lib.ttsp_nf4_gemm_splits(M, K, rows)
    assert rc == 0 and splits > 1
    ref = split_product(lin, x, splits, epi, r)
    nan = torch.isnan(ref.float())
    assert torch.equal(nan, torch.isnan(out.float())) and bool(nan.any()) and not bool(nan.all())
    assert torch.equal(out.view(torch.int16)[~nan], ref.view(torch.int16)[~nan])


@pytest.mark.gpu
def test_tile_gemm_is_reproducible(nf4):
    """Twenty runs of each form give the same bits (a stage refilled while
    another wave still reads it would not)."""
    for (M, K), rows in (((1542, 2688), 200), ((9728, 2560), 256), ((9728, 2560), 512)):
        lin = to_linear(random_layer(M, K, True, seed=3), torch.bfloat16)
        assert nf4.prepare(lin)
        x = from_bits(randn_bits(rows * K, torch.bfloat16, seed=4), torch.bfloat16).view(rows, K)
        first = nf4.matmul(lin, x).clone()
        for _ in range(20):
            assert torch.equal(nf4.matmul(lin, x).view(torch.int16), first.view(torch.int16))
