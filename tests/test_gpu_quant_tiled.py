"""GPU: the tiled W8A8 product (more rows than the few-row kernels take) bit for
bit against the oracle, at the edges of its 64 / 128 tiles, its 128-deep slabs
and its rings, for each tier, with the epilogue; and zero points beyond the
first entries, which the row quantizer's launch checks."""
import numpy as np
import pytest

from hologram_amd import DTYPE_E8CB, DTYPE_I4, DTYPE_I8, UnsupportedOp
from hologram_amd import fused_activation as FA
import test_gpu_quant as base

pytestmark = pytest.mark.gpu

import oracle  # noqa: E402

KW = dict(inner=1, bq_omajor=True, act_quant=1)
SHAPES = [  # m, k, n: tiles 64 x 64, 64 x 128, 128 x 128; slabs and rings whole and not
    (17, 128, 64), (65, 256, 100), (130, 384, 700), (64, 1152, 8200), (200, 2048, 5000),
    (1030, 640, 4100), (512, 8192, 136), (96, 160, 300), (70, 32, 65),
]


@pytest.mark.parametrize("tier", [DTYPE_I8, DTYPE_I4, DTYPE_E8CB])
@pytest.mark.parametrize("m,k,n", SHAPES)
def test_bit_exact(torch_cuda, backend, tier, m, k, n):
    rng = np.random.default_rng(m + k + n + tier)
    a, bq, scales, cb = base.w8a8_operands(rng, tier, m, k, n)
    a[3 * k] = np.nan                     # never the maximum, quantized to 0
    a[4 * k + 1] = np.inf                 # the row's scale
    kw = dict(m=m, k=k, n=n, channels=n, quant_dtype=tier, **KW)
    got = base.run_mmd(torch_cuda, backend, kw, a, bq, scales, np.zeros(n, np.int32), codebook=cb)
    assert base.same_bits(got, oracle.matmul_q_omajor(tier, a, bq, scales, m, k, n, codebook=cb))


@pytest.mark.parametrize("act,res", [(FA.GELU, True), (FA.SILU, False), (0, True), (FA.EXP, True)])
@pytest.mark.parametrize("m,n", [(70, 90), (200, 4500)])
def test_epilogue_bit_exact(torch_cuda, backend, m, n, act, res):
    k = 256
    rng = np.random.default_rng(act + 10 * res + m)
    a, bq, scales, _ = base.w8a8_operands(rng, DTYPE_I8, m, k, n)
    r = rng.standard_normal(m * n).astype(np.float32) if res else None
    kw = dict(m=m, k=k, n=n, channels=n, quant_dtype=DTYPE_I8, act=act, **KW)
    got = base.run_mmd(torch_cuda, backend, kw, a, bq, scales, np.zeros(n, np.int32), residual=r)
    want = oracle.matmul_q_omajor(DTYPE_I8, a, bq, scales, m, k, n)
    if res:
        want = (want + r).astype(np.float32)
    assert base.same_bits(got, oracle.fused_act_f32(act, want) if act else want)


@pytest.mark.parametrize("k", [64, 201])     # the vector and the general row quantizer
@pytest.mark.parametrize("at", [0, 1023, 1024, 5000])
def test_any_nonzero_zero_point_is_reported(torch_cuda, backend, k, at):
    m, n = 20, 5001
    rng = np.random.default_rng(at)
    a, bq, scales, _ = base.w8a8_operands(rng, DTYPE_I8, m, k, n)
    zps = np.zeros(n, np.int32)
    zps[at] = 1 << 24
    kw = dict(m=m, k=k, n=n, channels=n, quant_dtype=DTYPE_I8, **KW)
    with pytest.raises(UnsupportedOp):
        base.run_mmd(torch_cuda, backend, kw, a, bq, scales, zps)
    got = base.run_mmd(torch_cuda, backend, kw, a, bq, scales, np.zeros(n, np.int32))
    assert base.same_bits(got, oracle.matmul_q_omajor(DTYPE_I8, a, bq, scales, m, k, n))
