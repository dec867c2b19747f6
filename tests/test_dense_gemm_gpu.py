"""The two-launch NF4 product of long prompts (csrc/nf4_gemm_dense.hip):
dequantise into a workspace, then the dense matrix kernel, against the fp64
product; its SwiGLU pair against its two launches."""

import numpy as np
import pytest
import torch

from oracle import oracle as o
from tests.conftest import beyond_rounding_error
from tests.gpuutil import bits, dt_code, from_bits, randn_bits
from tests.nf4data import oracle_args, random_layer, to_linear


@pytest.fixture(scope="module")
def nf4():
    from ttspipe_amd import nf4gemv

    assert nf4gemv.install()
    return nf4gemv


def _plan(M, K, rows):
    from ttspipe_amd import _lib

    return _lib.load().ttsp_nf4_gemm_dense_splits(M, K, rows)


def test_dense_plan_covers_long_prompts_only():
    """Not up to 512 rows, not small products, not byte offsets of 2^31; else
    unsplit or the 512-row plan's splits."""
    from ttspipe_amd import _lib

    assert _plan(9728, 2560, 512) == 0 and _plan(1024, 1024, 1024) == 0 and _plan(4096, 2560, 1 << 20) == 0
    assert _plan(1 << 17, 1 << 14, 1024) == 0
    for M, K in ((9728, 2560), (2560, 9728), (2560, 4096), (6144, 2560), (9730, 2560), (4096, 1024), (128, 32768)):
        for rows in (513, 700, 800, 1024, 1500, 2048, 5000):
            sp = _plan(M, K, rows)
            assert sp in (0, 1, _lib.load().ttsp_nf4_gemm_splits(M, K, 512))
            assert sp or rows < 1024 or M * K < 1 << 21 or M * K * rows < 2.5e9
            assert sp < 2 or M % 4 == 0


def test_dense_form_only_where_it_pays():
    """`ttsp_nf4_gemm_dense_pays`: large weights over many rows, not the small
    ones whose tiles are faster (1024 x 3072 at 2048 rows 26 against 38 us), and
    never where the form does not serve; below 1024 rows served means paying."""
    from ttspipe_amd import _lib

    pays = _lib.load().ttsp_nf4_gemm_dense_pays
    for M, K, rows in ((9728, 2560, 1024), (9728, 2560, 2048), (6144, 2560, 2048), (2560, 9728, 2048), (2560, 9728, 800)):
        assert pays(M, K, rows) == 1
    for M, K, rows in ((1024, 3072, 1024), (1024, 3072, 2048), (1536, 2560, 1024), (2048, 2048, 1024), (3072, 1024, 1200),
                       (9728, 2560, 600), (512, 512, 2048), (9728, 2560, 512)):
        assert pays(M, K, rows) == 0
    for M in (256, 1024, 1540, 4096, 9730):
        for K in (512, 1024, 2560, 4096):
            for rows in (513, 700, 1023, 1024, 1500, 3000):
                sp = _plan(M, K, rows)
                assert pays(M, K, rows) <= (sp > 0) and (rows >= 1024 or pays(M, K, rows) == (sp > 0))


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1024, 1500])
def test_matmul_takes_the_dense_form_where_it_pays(nf4, rows):
    """A small weight's rows run the tiles unless the caller keeps the merged
    spans' order (`wide`); both within the bar of each other's rounding."""
    from ttspipe_amd import _lib

    M, K = 1024, 3072
    lib, lin = _lib.load(), to_linear(random_layer(M, K, True, seed=9), torch.bfloat16)
    assert nf4.prepare(lin) and _plan(M, K, rows) and not lib.ttsp_nf4_gemm_dense_pays(M, K, rows)
    x = from_bits(randn_bits(rows * K, torch.bfloat16, seed=3), torch.bfloat16).view(rows, K)
    fast, out = lin._nf4_fast, torch.empty(rows, M, dtype=torch.bfloat16, device="cuda")
    splits = lib.ttsp_nf4_gemm_tile_splits(M, K, rows)
    work = torch.empty(splits * rows * M, device="cuda")
    rc = lib.ttsp_nf4_gemm_split(x.data_ptr(), _lib.DT_BF16, fast["w"], fast["a8"], fast["amax"], fast["code2"],
                                 fast["offset"], fast["lut"].data_ptr(), out.data_ptr(), 0, 0, M, K, rows, 64, 256,
                                 work.data_ptr(), splits, _lib.stream())
    assert rc == 0 and torch.equal(nf4.matmul(lin, x), out)
    wide = nf4.matmul(lin, x, wide=True)
    assert float((wide.float() - out.float()).norm() / out.float().norm()) < 2**-8


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,rows", [(9728, 2560, 1100), (2560, 9728, 1100)])
def test_without_room_for_the_workspace_the_tiles_run(nf4, monkeypatch, M, K, rows):
    """A product whose dequantised weight does not fit the memory left runs the
    kernels that read the codes in place (the pair as two launches): within the
    roundings of the dense form, through the same calls."""
    lin, lin3 = (to_linear(random_layer(M, K, True, seed=s), torch.bfloat16) for s in (1, 2))
    assert nf4.prepare(lin) and nf4.prepare(lin3) and _plan(M, K, rows)
    x = from_bits(randn_bits(rows * K, torch.bfloat16, seed=3), torch.bfloat16).view(rows, K)
    dense, pair = nf4.matmul(lin, x), nf4.matmul_swiglu(lin, lin3, x)
    empty = torch.empty

    def limited(*size, **kw):
        if kw.get("dtype") is torch.uint8:
            raise torch.OutOfMemoryError("no room")
        return empty(*size, **kw)

    monkeypatch.setattr(torch, "empty", limited)
    tiles = nf4.matmul(lin, x)
    assert float((tiles.float() - dense.float()).norm() / dense.float().norm()) < 2**-8
    assert nf4.matmul_swiglu(lin, lin3, x) is None
    if pair is not None:
        two = nf4.matmul(lin3, x, epi=nf4.EPI_SILU_GATE, operand=tiles)
        assert float((two.float() - pair.float()).norm() / pair.float().norm()) < 2**-7


@pytest.mark.gpu
@pytest.mark.parametrize("shape,rows,splits,nested,dtype,epi", [
    ((9728, 2560), 1025, 1, True, torch.bfloat16, 0),    # one activation row in the last tile
    ((9730, 2560), 900, 1, False, torch.float16, 0),     # M % 4 == 2: element-wise stores
    ((9730, 2560), 900, 1, True, torch.bfloat16, 1),     # and element-wise residual reads
    ((6144, 2560), 2048, 1, True, torch.bfloat16, 0),    # 192 x 256 tiles, two runs of K
    ((6150, 2560), 2047, 1, False, torch.float16, 2),    # the same, ragged both ways
    ((2560, 9728), 1000, 4, True, torch.bfloat16, 1),    # K splits, the reduce's epilogue
    ((2564, 8192), 1030, 4, False, torch.float16, 2),    # M % 8 == 4 under a split
    ((2564, 8192), 1600, 1, True, torch.float16, 1),     # four runs of K in a workgroup
    ((1540, 9600), 1300, 1, True, torch.float16, 0),     # 150 K-steps
    ((4096, 1024), 4000, 1, True, torch.bfloat16, 0),    # 16 K-steps
])
def test_dense_gemm_against_fp64(nf4, orc, shape, rows, splits, nested, dtype, epi):
    """Rows past N and weight rows past M repeat the last ones and must not be
    stored; within the 2e-3 bar beyond the output's own rounding (fp32 sums of
    K products, as the fused kernels)."""
    (M, K), dt = shape, dt_code(dtype)
    assert _plan(M, K, rows) == splits
    layer = random_layer(M, K, nested, seed=M + rows)
    lin = to_linear(layer, dtype)
    assert nf4.prepare(lin)
    xb = randn_bits(rows * K, dtype, seed=rows, scale=0.5)
    x = from_bits(xb, dtype).view(rows, K)
    rb = randn_bits(rows * M, dtype, seed=5)
    guard = torch.full((rows + 1, M), 7.0, dtype=dtype, device="cuda")
    y = nf4.matmul(lin, x, epi=epi, operand=from_bits(rb, dtype).view(rows, M) if epi else None, out=guard[:rows],
                   wide=True)
    assert bool((guard[rows] == 7.0).all())
    sample = np.unique(np.r_[0:rows:61, rows - 1])
    ref = orc.nf4_gemm_ref(xb.reshape(rows, K)[sample], dt, **oracle_args(layer), M=M, K=K, N=sample.size, bs=64,
                           bs2=256).astype(np.float64).reshape(sample.size, M)
    if epi:
        ref = o.to_f32(o.from_f32(ref.astype(np.float32), dt), dt).astype(np.float64)
        r = o.to_f32(rb, dt).astype(np.float64).reshape(rows, M)[sample]
        silu = o.to_f32(o.from_f32((r / (1 + np.exp(-r))).astype(np.float32), dt), dt).astype(np.float64)
        ref = r + ref if epi == 1 else silu * ref
    got = o.to_f32(bits(y), dt).reshape(rows, M)[sample]
    assert beyond_rounding_error(got, ref, dt) < 2e-3


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,rows,nested,dtype", [(9728, 2560, 1300, True, torch.bfloat16),
                                                   (4096, 1024, 4000, False, torch.float16),
                                                   (2562, 2688, 2100, True, torch.bfloat16)])
def test_dense_swiglu_pair_equals_its_two_launches(nf4, M, K, rows, nested, dtype):
    from ttspipe_amd import _lib

    w1 = to_linear(random_layer(M, K, nested, seed=1), dtype)
    w3 = to_linear(random_layer(M, K, nested, seed=2), dtype)
    assert nf4.prepare(w1) and nf4.prepare(w3)
    x = from_bits(randn_bits(rows * K, dtype, seed=3), dtype).view(rows, K)
    assert _lib.load().ttsp_nf4_gemm_dense_swiglu_fits(M, K, rows) == 1
    two = nf4.matmul(w3, x, epi=nf4.EPI_SILU_GATE, operand=nf4.matmul(w1, x))
    one = nf4.matmul_swiglu(w1, w3, x)
    assert one is not None and torch.equal(one.view(torch.int16), two.view(torch.int16))
