"""GPU parity of the tiled prompt attention over the int8 cache (op 125, bf16
rows, head_dim 64 and 128) for every kind of group, at rows, keys and buckets
off its 128-row and 64-key tiles: within 1e-2 of the oracle's row, as the op's
other forms; rows that see no key exactly zero; one cache row whose scales are
NaN leaves the rows that do not see it untouched."""
import numpy as np
import pytest

import oracle
from conftest import from_dev, to_dev
from hologram_amd import (DTYPE_BF16, DTYPE_F32, AttentionI8RowsCall, BufferRef, DecodeAttentionI8Call,
                          DeviceWorkspace, KernelCall, UnsupportedOp)
from test_gpu_prefill import make_cache, run_rows

pytestmark = pytest.mark.gpu

CASES = [  # B, T, H, Hkv, D, S, lens: the first seven have 1024 packed workgroups or more
    (32, 65, 8, 8, 64, 100, [65, 100, 20, 3] * 8),   # G 1
    (40, 70, 6, 2, 128, 200, [70, 133] * 20),        # G 3: a row's heads straddle waves
    (64, 9, 64, 8, 64, 64, [63, 9] * 32),            # G 8, 72 rows
    (32, 17, 32, 2, 128, 100, [90, 5] * 16),         # G 16, 272 rows
    (4, 70, 8, 4, 128, 4096, [3000, 70, 2100, 64]),  # a bucket of more than one chunk
    (64, 129, 4, 1, 128, 192, [192, 129] * 32),      # one row past four tiles
    (128, 2, 64, 8, 64, 64, [64, 1] * 64),           # two rows
    (2, 33, 4, 1, 128, 192, [192, 33]),              # few: packed
    (1, 20, 8, 2, 64, 4096, [3000]),                 # few, chunks
    (1, 64, 20, 1, 64, 128, [64]),                   # G 20: the general kernel
]


@pytest.mark.parametrize("B,T,H,Hkv,D,S,lens", CASES)
def test_prompt_tiles_parity(torch_cuda, backend, B, T, H, Hkv, D, S, lens):
    got, want, _ = run_rows(torch_cuda, backend, B, T, H, Hkv, D, S, lens, seed=T + S + D)
    for b in range(B):
        for t in range(T):
            if lens[b] - (T - 1 - t) <= 0:
                assert np.all(got[b, t] == 0), (b, t)
            else:
                err = np.max(np.abs(got[b, t] - want[b, t])) / (np.max(np.abs(want[b, t])) + 1e-9)
                assert err <= 1e-2, (b, t, err)


@pytest.mark.parametrize("B,T,H,Hkv,D,S", [(32, 65, 8, 8, 64, 100), (2, 33, 4, 1, 128, 192),
                                           (1, 20, 8, 2, 64, 4096), (1, 64, 20, 1, 64, 128)])
def test_a_length_past_the_bucket_is_reported_by_every_form(torch_cuda, backend, B, T, H, Hkv, D, S):
    """One sequence, the last, one key past the bucket: tiled, packed, chunked
    and general form each raise it, and the flag is clear afterwards."""
    with pytest.raises(UnsupportedOp):
        run_rows(torch_cuda, backend, B, T, H, Hkv, D, S, [S] * (B - 1) + [S + 1], seed=1)
    backend.synchronize()
    run_rows(torch_cuda, backend, B, T, H, Hkv, D, S, [S] * B, seed=1)


@pytest.mark.parametrize("D", [64, 128])
def test_scales_of_unseen_rows_do_not_reach_earlier_rows(torch_cuda, backend, D):
    """Scales from 2^-20 to 2^20 in one cache; the last visible row's are NaN,
    which only the last query row sees, and rows past it hold infinities."""
    B, T, H, Hkv, S, n = 1, 70, 512, 256, 200, 150
    rng = np.random.default_rng(D)
    kq, ks = make_cache(rng, Hkv, S, D)
    vq, vs = make_cache(rng, Hkv, S, D)
    ks, vs = (np.array(x).view(np.float32).reshape(Hkv, S).copy() for x in (ks, vs))
    vs[:, 30] *= 2.0 ** 20
    vs[:, 31] *= 2.0 ** -20
    vs[:, 130] *= 2.0 ** 21
    want_vs = vs.copy()
    for x in (ks, vs):
        x[:, n - 1], x[:, n:] = np.nan, np.inf
    q32 = rng.standard_normal(B * T * H * D).astype(np.float32)
    qb = (q32.view(np.uint32) >> 16).astype(np.uint16)
    q32 = (qb.astype(np.uint32) << 16).view(np.float32)
    lens = np.array([n], np.uint32)
    ws = DeviceWorkspace()
    for s, a in enumerate([qb, kq, vq, ks, vs, lens]):
        ws.bind(s, to_dev(torch_cuda, a))
    out = torch_cuda.zeros(B * T * H * D * 2, dtype=torch_cuda.uint8, device="cuda")
    ws.bind(6, out)
    attn = DecodeAttentionI8Call(*[BufferRef(i) for i in range(7)], B, H, Hkv, S, D, 0, DTYPE_BF16)
    backend.dispatch(KernelCall.AttentionI8Rows(AttentionI8RowsCall(attn, T)), ws)
    backend.synchronize()
    got = (from_dev(out, np.uint16).astype(np.uint32) << 16).view(np.float32).reshape(T, H, D)
    ks_ok = np.where(np.isfinite(ks), ks, 0.02).astype(np.float32)
    want = oracle.attention_i8_rows(q32, kq, ks_ok, vq, want_vs, lens, B, T, H, Hkv, S, D,
                                    oracle.attn_scale(D)).reshape(T, H, D)
    seen = slice(0, T - 1)
    err = np.abs(got[seen] - want[seen]).max(-1) / (np.abs(want[seen]).max(-1) + 1e-9)
    assert np.isfinite(got[seen]).all() and err.max() <= 1e-2


@pytest.mark.parametrize("H,Hkv,S", [(512, 128, 200), (8, 2, 200), (8, 2, 4096)])   # tiled, packed, chunks
@pytest.mark.parametrize("D", [64, 128])
def test_a_row_leaves_the_others_alone_whatever_it_holds(torch_cuda, backend, D, H, Hkv, S):
    """Query rows of NaN, infinities and values to 1e30, some seeing keys and some
    none, among N(0, 1) rows and rows 16 times as large, all in one tile: every
    other row stays within the bound, and the rows that see no key are zeros. Some
    v-scales are negative; in the tiled form one that only the last token sees is
    infinite."""
    B, T, n = 1, 70, 64
    rng = np.random.default_rng(D + 1)
    kq, ks = make_cache(rng, Hkv, S, D)
    vq, vs = make_cache(rng, Hkv, S, D)
    ks, vs = (np.array(x).view(np.float32).reshape(Hkv, S).copy() for x in (ks, vs))
    vs[:, ::3] *= -1.0
    vs[:, 6] *= 300.0      # negative, and past f16 at the exponent of the positive ones
    want_vs = vs.copy()
    if H == 512:
        vs[:, n - 1] = np.inf
    q32 = rng.standard_normal((T, H, D)).astype(np.float32)
    q32[40:48] *= 16.0
    odd = {0: np.nan, 2: 1e30, 3: np.inf, 20: np.nan, 30: 1e30, 33: -np.inf}   # 0..5 see no key
    for t, v in odd.items():
        q32[t, 0::4, ::7] = v
    qb = (q32.view(np.uint32) >> 16).astype(np.uint16)
    q32 = (qb.astype(np.uint32) << 16).view(np.float32)
    got, _ = _rows_over(torch_cuda, backend, qb, kq, vq, ks, vs, n, T, H, Hkv, S, D)
    clean = np.ones((T, H), bool)
    for t in odd:
        clean[t, 0::4] = False
    clean[T - 1] = False
    clean[:T - n] = False
    want = oracle.attention_i8_rows(np.where(np.isfinite(q32), q32, 0).astype(np.float32).ravel(), kq, ks, vq,
                                    want_vs, np.array([n], np.uint32), B, T, H, Hkv, S, D,
                                    oracle.attn_scale(D)).reshape(T, H, D)
    assert np.all(got[:T - n] == 0)
    err = np.abs(got[clean] - want[clean]).max(-1) / (np.abs(want[clean]).max(-1) + 1e-9)
    assert np.isfinite(got[clean]).all() and err.max() <= 1e-2


def _rows_over(torch, backend, qb, kq, vq, ks, vs, n, T, H, Hkv, S, D):
    ws = DeviceWorkspace()
    for s, a in enumerate([qb.ravel(), kq, vq, ks, vs, np.array([n], np.uint32)]):
        ws.bind(s, to_dev(torch, a))
    out = torch.zeros(T * H * D * 2, dtype=torch.uint8, device="cuda")
    ws.bind(6, out)
    attn = DecodeAttentionI8Call(*[BufferRef(i) for i in range(7)], 1, H, Hkv, S, D, 0, DTYPE_BF16)
    backend.dispatch(KernelCall.AttentionI8Rows(AttentionI8RowsCall(attn, T)), ws)
    backend.synchronize()
    return (from_dev(out, np.uint16).astype(np.uint32) << 16).view(np.float32).reshape(T, H, D), out


@pytest.mark.parametrize("S", [256, 4096])   # packed, chunks
def test_64_dim_rows_keep_q_exact_where_they_are_few(torch_cuda, backend, S):
    """Channel 0 of Q is 2^13 times the others and meets keys that are 0 there, so
    the scores are the other channels' alone: a Q of 15 bits would round those to
    whole steps of 1 and miss by half the result; of 23 bits, the result is the
    oracle's within the truncation (bound 1e-2, as above)."""
    T, H, Hkv, D, n = 24, 8, 2, 64, 200
    rng = np.random.default_rng(S)
    x = rng.standard_normal((Hkv, S, D)).astype(np.float32)
    x[:, :, 0] = 0.0
    zero = lambda: (np.zeros(Hkv * S * D, np.int8), np.zeros(Hkv * S, np.float32))  # noqa: E731
    kq, ks = oracle.kv_quant_append(x, DTYPE_F32, 0, *zero(), Hkv, S, S, D)
    vq, vs = make_cache(rng, Hkv, S, D)
    q32 = rng.standard_normal((T, H, D)).astype(np.float32)
    q32[:, :, 0] = 8192.0
    qb = (q32.view(np.uint32) >> 16).astype(np.uint16)
    q32 = (qb.astype(np.uint32) << 16).view(np.float32)
    got, _ = _rows_over(torch_cuda, backend, qb, kq, vq, ks, vs, n, T, H, Hkv, S, D)
    want = oracle.attention_i8_rows(q32.ravel(), kq, ks, vq, vs, np.array([n], np.uint32), 1, T, H, Hkv, S, D,
                                    oracle.attn_scale(D)).reshape(T, H, D)
    err = np.abs(got - want).max(-1) / (np.abs(want).max(-1) + 1e-9)
    assert err.max() <= 1e-2
