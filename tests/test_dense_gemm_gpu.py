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
    y = nf4.matmul(lin, x, epi=epi, operand=from_bits(rb, dtype).view(rows, M) if epi else None, out=guard[:rows])
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
