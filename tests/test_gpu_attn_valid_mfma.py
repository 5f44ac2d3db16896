"""GPU parity of DecodeAttentionValid (121) and its mask form (119) on the
matrix-core kernels, at the sizes where their tiles, lists and operands end:
rows and keys off every tile edge, head_dim off the 32-dim blocks, empty past,
nothing realized, lists shared among workgroups; and the values they must carry
as the scalar walk does (NaN and Inf in V and K, masks of the lowest f32).

Bounds. bf16 / f16 outputs: 1e-2 of the row's largest value, as for the scalar
kernels (the narrowing is 2^-8 / 2^-11 of a value). f32: 1e-5 of the f64 law.
Non-finite outputs: exactly where the oracle has them."""
import numpy as np
import pytest

import oracle
from conftest import to_dev
from hologram_amd import (DTYPE_BF16, DTYPE_F16, DTYPE_F32, BufferRef, DecodeAttentionCall,
                          DecodeAttentionValidCall, DeviceWorkspace, HipBackend, KernelCall)
from test_gpu_attn_mask import run_mask
from test_gpu_attn_valid import TOL, dec, enc, law_f64, row_err, run_valid

pytestmark = pytest.mark.gpu

SHAPES = [  # b, h, hkv, m, past, valid, d
    (1, 4, 1, 33, 200, 130, 128),    # 132 rows: a full tile and four rows
    (2, 8, 2, 65, 64, 64, 64),       # 260 rows, a past of exactly one tile
    (1, 2, 2, 127, 0, 0, 96),        # no past, one head per tile
    (1, 6, 2, 40, 300, 0, 80),       # nothing realized
    (1, 8, 1, 3, 1000, 999, 128),    # 24 rows: the list shared among workgroups
    (1, 1, 1, 129, 63, 63, 72),      # one head; rows, keys and dims off every edge
    (2, 4, 4, 20, 65, 77, 8),        # the narrowest rows; valid beyond the bucket
]


@pytest.mark.parametrize("dtype", [DTYPE_BF16, DTYPE_F16])
@pytest.mark.parametrize("b,h,hkv,m,past,valid,d", SHAPES)
def test_rows_parity(torch_cuda, backend, b, h, hkv, m, past, valid, d, dtype):
    got, want, _ = run_valid(torch_cuda, backend, b, h, hkv, m, past, valid, d, dtype, seed=m + past + d)
    assert np.all(np.isfinite(got))
    err = row_err(got, want)
    assert err <= TOL[dtype], f"normalized error {err:.3g}"


@pytest.mark.parametrize("dtype", [DTYPE_BF16, DTYPE_F16])
@pytest.mark.parametrize("kind", ["realized", "random"])
@pytest.mark.parametrize("b,h,hkv,m,past,new,d", [
    (1, 4, 1, 33, 131, 33, 128), (1, 8, 2, 50, 64, 0, 64), (2, 2, 1, 40, 0, 70, 80),
    (1, 8, 1, 4, 2000, 4, 96)])
def test_rows_mask_parity(torch_cuda, backend, b, h, hkv, m, past, new, d, kind, dtype):
    got, want, _, mask = run_mask(torch_cuda, backend, b, h, hkv, m, past, new, d, dtype, kind,
                                  seed=m + past + new + d)
    assert np.all(np.isfinite(got))
    erased = ~np.isfinite(mask).any(axis=1)
    assert not got.reshape(b, h, m, d)[:, :, erased].any()
    assert row_err(got, want) <= TOL[dtype]


FEW = [     # b, h, hkv, m, past, valid, d: up to 16 rows a plane (f32: any)
    (1, 16, 1, 1, 700, 650, 128),    # 16 rows of one plane, several shares
    (3, 3, 3, 1, 31, 31, 64),        # one row; past and list off the 32-key block
    (2, 8, 4, 7, 0, 0, 96),          # no past
    (1, 5, 1, 3, 129, 128, 40),      # 15 rows; head_dim off the 64-byte steps
    (1, 4, 4, 1, 5000, 1, 8),        # one realized key of many: most shares empty
    (1, 4, 2, 20, 100, 90, 72),      # 40 rows: f32 in three row tiles
    (64, 8, 8, 1, 40, 40, 128),      # 512 planes: no merge
]


@pytest.mark.parametrize("dtype", [DTYPE_BF16, DTYPE_F16, DTYPE_F32])
@pytest.mark.parametrize("b,h,hkv,m,past,valid,d", FEW)
def test_few_rows_parity(torch_cuda, backend, b, h, hkv, m, past, valid, d, dtype):
    f32 = dtype == DTYPE_F32
    got, want, law = run_valid(torch_cuda, backend, b, h, hkv, m, past, valid, d, dtype,
                               seed=m + past + d + h, with_law=f32)
    assert np.all(np.isfinite(got))
    assert row_err(got, law if f32 else want) <= TOL[dtype]


def dispatch(torch, backend, make, wrap, ops, last, shape, dtype, shift=0):
    """shift: bytes the operands lie past 16-byte alignment (4: the element-wise form)."""
    b, h, hkv, m, past, new, d = shape
    es = 4 if dtype == DTYPE_F32 else 2
    ws = DeviceWorkspace()
    for s, x in enumerate(ops + [last]):
        t = to_dev(torch, x) if x.size else torch.zeros(64, dtype=torch.uint8, device="cuda")
        if shift:
            t = torch.cat([torch.zeros(shift, dtype=torch.uint8, device="cuda"), t.view(torch.uint8)])[shift:]
        ws.bind(s, t)
    out = torch.full((b * h * m * d * es,), 0x55, dtype=torch.uint8, device="cuda")
    ws.bind(6, out)
    backend.dispatch(wrap(make(*[BufferRef(s) for s in range(7)], b, h, hkv, m, past, new, d, 0,
                               dtype)), ws)
    backend.synchronize()
    return dec(out.cpu().numpy().view(np.float32 if es == 4 else np.uint16), dtype).reshape(b, h, m, d)


def same_values(got, want, tol):
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.isposinf(got), np.isposinf(want))
    assert np.array_equal(np.isneginf(got), np.isneginf(want))
    fin = np.isfinite(want)
    scale = np.max(np.abs(np.where(fin, want, 0)), axis=-1, keepdims=True) + 1e-9
    assert np.max(np.where(fin, np.abs(np.where(fin, got, 0) - np.where(fin, want, 0)), 0) / scale) <= tol


@pytest.mark.parametrize("dtype", [DTYPE_BF16, DTYPE_F16, DTYPE_F32])
@pytest.mark.parametrize("b,h,hkv,m,past,valid,d,where", [
    (2, 4, 2, 5, 100, 90, 64, "new"), (1, 16, 1, 1, 700, 650, 128, "past"),
    (1, 4, 4, 1, 50, 40, 40, "keys"),
    (1, 4, 2, 40, 100, 90, 64, "new"),     # late new rows: earlier query rows do not see them
    (1, 4, 2, 40, 100, 90, 64, "past"),
    (1, 8, 1, 3, 1500, 1400, 128, "past"), # one share of several
    (1, 4, 2, 40, 100, 90, 64, "keys"),    # NaN and Inf scores: a NaN score weighs 0
    (1, 6, 1, 33, 200, 130, 128, "past"),  # 198 rows in fours, the last two short; keys past 64
    (1, 4, 2, 40, 100, 90, 72, "new"),     # an odd count of 16-byte chunks
    (2, 3, 1, 1, 300, 299, 40, "past"),    # three rows
])
def test_non_finite_operands(torch_cuda, backend, b, h, hkv, m, past, valid, d, where, dtype):
    rng = np.random.default_rng(3)
    n = (b * h * m * d, b * hkv * past * d, b * hkv * past * d, b * hkv * m * d, b * hkv * m * d)
    q, kp, vp, kn, vn = (rng.standard_normal(k).astype(np.float32) for k in n)
    if where == "new":
        v = vn.reshape(b, hkv, m, d)
        v[:, :, m - 2, ::2], v[:, :, m - 1, 1::2], v[:, :, m // 2, 3] = np.nan, np.inf, -np.inf
    elif where == "past":
        v = vp.reshape(b, hkv, past, d)
        v[:, :, 7, 1], v[:, :, valid - 1, 2], v[:, :, 7, 5] = np.inf, np.nan, -np.inf
    else:
        kp.reshape(b, hkv, past, d)[:, :, 11, 0] = np.nan
        kp.reshape(b, hkv, past, d)[:, 0, 12, 0] = np.inf
    ops = [enc(x, dtype) for x in (q, kp, vp, kn, vn)]
    shape = (b, h, hkv, m, past, m, d)
    got = dispatch(torch_cuda, backend, DecodeAttentionValidCall, KernelCall.DecodeAttentionValid, ops,
                   np.array([valid], np.uint32), shape, dtype)
    want = dec(oracle.decode_attention_valid(*ops, valid, b, h, hkv, m, past, m, d, 0, dtype),
               dtype).reshape(b, h, m, d)
    if where != "keys":
        assert not np.isfinite(want).all()
    same_values(got, want, TOL[dtype])


@pytest.mark.parametrize("dtype", [DTYPE_BF16, DTYPE_F16, DTYPE_F32])
@pytest.mark.parametrize("h,m", [(4, 40), (4, 1)])
def test_mask_of_the_lowest_value_and_erased_non_finite_v(torch_cuda, backend, h, m, dtype):
    """A row masked by the lowest f32 everywhere weighs every key alike; an
    erased (-inf) key's NaN V still reaches the output (0 * NaN)."""
    b, hkv, past, d = 1, 1, 70, 64
    rng = np.random.default_rng(4)
    ops = [enc(rng.standard_normal(k), dtype) for k in
           (b * h * m * d, past * d, past * d, m * d, m * d)]
    mask = np.zeros((m, past + m), np.float32)
    mask[0] = np.finfo(np.float32).min
    mask[m // 2, 5:] += -1e30
    mask[m - 1, 30:] = -np.inf
    shape = (b, h, hkv, m, past, m, d)
    args = (torch_cuda, backend, DecodeAttentionCall, KernelCall.DecodeAttention)
    for vnan in (False, True):
        if vnan:
            ops[2] = ops[2].copy()
            ops[2].reshape(past, d)[60, 9] = {DTYPE_BF16: 0x7FC0, DTYPE_F16: 0x7E00, DTYPE_F32: np.nan}[dtype]
        got = dispatch(*args, ops, mask.ravel(), shape, dtype)
        want = dec(oracle.decode_attention(*ops, mask, b, h, hkv, m, past, m, d, 0, dtype),
                   dtype).reshape(b, h, m, d)
        same_values(got, want, TOL[dtype])


@pytest.mark.parametrize("dtype", [DTYPE_BF16, DTYPE_F16, DTYPE_F32])
@pytest.mark.parametrize("b,h,hkv,m,past,new,d", [(1, 4, 1, 33, 131, 30, 128), (2, 8, 2, 1, 700, 45, 64)])
def test_mask_form_split_equals_precatenated(torch_cuda, backend, b, h, hkv, m, past, new, d, dtype):
    """Past and new rows form one list: where they part changes no bit."""
    rng = np.random.default_rng(6)
    q = enc(rng.standard_normal(b * h * m * d), dtype)
    k, v = (enc(rng.standard_normal(b * hkv * (past + new) * d), dtype).reshape(b * hkv, past + new, d)
            for _ in range(2))
    mask = (rng.standard_normal((m, past + new)) * 2).astype(np.float32)
    mask[rng.random(mask.shape) < 0.3] = -np.inf
    outs = []
    for cut in (past, past + new, 64):
        ops = [q] + [np.ascontiguousarray(x).ravel() for x in
                     (k[:, :cut], v[:, :cut], k[:, cut:], v[:, cut:])]
        outs.append(dispatch(torch_cuda, backend, DecodeAttentionCall, KernelCall.DecodeAttention, ops,
                             mask.ravel(), (b, h, hkv, m, cut, past + new - cut, d), dtype))
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))
    assert np.array_equal(outs[0].view(np.uint32), outs[2].view(np.uint32))


def test_capture_on_a_backend_that_has_no_scratch(torch_cuda):
    """A call that the element-wise form splits nowhere needs no scratch, so it
    can be captured on a fresh backend, and later growth does not touch its
    replays."""
    torch = torch_cuda
    b, h, hkv, d, m, past = 1, 32, 8, 128, 300, 1537
    g = torch.Generator(device="cuda")
    g.manual_seed(m)
    mk = lambda rows, heads: torch.randn((b * heads * rows, d), generator=g, device="cuda").to(torch.bfloat16)
    ops = [mk(m, h), mk(past, hkv), mk(past, hkv), mk(m, hkv), mk(m, hkv),
           torch.tensor([past], dtype=torch.int32, device="cuda")]
    out = torch.zeros((b * h * m, d), dtype=torch.bfloat16, device="cuda")
    ws = DeviceWorkspace()
    for s, x in enumerate(ops + [out]):
        ws.bind(s, x)
    call = KernelCall.DecodeAttentionValid(DecodeAttentionValidCall(
        *[BufferRef(s) for s in range(7)], b, h, hkv, m, past, m, d, 0, DTYPE_BF16))
    stream = torch.cuda.Stream()
    be = HipBackend(stream=stream.cuda_stream)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        be.dispatch(call, ws)
    graph.replay()
    torch.cuda.synchronize()
    captured = out.float().cpu().numpy()
    be.dispatch(call, ws)                       # eager: takes scratch now
    be.synchronize()
    eager = out.float().cpu().numpy()
    assert row_err(captured, eager) <= TOL[DTYPE_BF16]
    for _ in range(2):
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(out.float().cpu().numpy(), captured)
    be.close()


@pytest.mark.parametrize("mask,b,h,hkv,past,valid,new,d", [
    (True, 2, 4, 4, 80, 8, 1, 128), (True, 1, 8, 2, 70, 14, 23, 80), (True, 8, 64, 8, 227, 13, 1, 128),
    (False, 1, 16, 8, 85, 4, 9, 64)])
def test_f32_is_no_further_from_64_bits_than_the_element_wise_form(torch_cuda, backend, mask, b, h, hkv, past,
                                                                   valid, new, d):
    """Over few keys, where no sum is long: the distance from 64 bits, as the
    geometric mean of 30 draws' ratios, against the element-wise form's (operands
    4 bytes off alignment take it). One draw's ratio scatters by 5% over few rows,
    the mean of 30 by 1%; it is 0.86-0.97, and was 1.00-1.035 with the scores in four sums."""
    ratios = []
    for seed in range(30):
        rng = np.random.default_rng(seed)
        q, kp, vp, kn, vn = (rng.standard_normal(k).astype(np.float32) for k in (
            (b, h, new, d), (b, hkv, past, d), (b, hkv, past, d), (b, hkv, new, d), (b, hkv, new, d)))
        j, i = np.arange(past + new), np.arange(new)[:, None]
        seen = (j < valid) | ((j >= past) & (j <= past + i))
        k, v = (np.repeat(np.concatenate(x, 2).astype(np.float64), h // hkv, 1) for x in ((kp, kn), (vp, vn)))
        w = np.where(seen, np.einsum("bhid,bhjd->bhij", q.astype(np.float64), k) / np.sqrt(d), -np.inf)
        w = np.exp(w - w.max(-1, keepdims=True))
        want = np.einsum("bhij,bhjd->bhid", w / w.sum(-1, keepdims=True), v)
        make, wrap = ((DecodeAttentionCall, KernelCall.DecodeAttention) if mask else
                      (DecodeAttentionValidCall, KernelCall.DecodeAttentionValid))
        last = np.where(seen, 0, -np.inf).astype(np.float32).ravel() if mask else np.array([valid], np.uint32)
        err = [np.linalg.norm(dispatch(torch_cuda, backend, make, wrap, [x.ravel() for x in (q, kp, vp, kn, vn)], last,
                                       (b, h, hkv, new, past, new, d), DTYPE_F32, shift) - want) for shift in (0, 4)]
        ratios.append(err[0] / err[1])
    assert np.exp(np.mean(np.log(ratios))) <= 1.0


@pytest.mark.parametrize("b,m,past", [(2, 509, 1537), (1, 64, 200)])
def test_a_non_finite_v_costs_no_more_than_the_general_form(torch_cuda, backend, b, m, past):
    """An infinity in V sends a prompt's shares to the scalar walk: within twice
    the general form's time on the same call (its operands 4 bytes off alignment;
    measured 2.8 against 3.9 ms, 65 against 57 us; 32 and 4 ms before the walk took
    its rows in fours, 0.4 ms with a tile's rows in one workgroup)."""
    torch, h, hkv, d = torch_cuda, 32, 8, 128
    g = torch.Generator(device="cuda")
    g.manual_seed(0)
    shapes = [(b * h * m, d), (b * hkv * past, d), (b * hkv * past, d), (b * hkv * m, d), (b * hkv * m, d)]
    ops = [torch.randn(x, generator=g, device="cuda").to(torch.bfloat16) for x in shapes]
    ops[2].view(b * hkv, past, d)[:, 5, 3] = float("inf")
    valid = torch.tensor([past], dtype=torch.int32, device="cuda")
    call = KernelCall.DecodeAttentionValid(DecodeAttentionValidCall(
        *[BufferRef(s) for s in range(7)], b, h, hkv, m, past, m, d, 0, DTYPE_BF16))
    took = []
    for shift in (0, 2):
        ws, kept = DeviceWorkspace(), []
        for s, x in enumerate(ops + [valid, torch.zeros_like(ops[0])]):
            x = x.reshape(-1)
            kept.append(torch.cat([torch.zeros(shift, dtype=x.dtype, device="cuda"), x])[shift:] if s not in (5,) else x)
            ws.bind(s, kept[-1])
        times = []
        for _ in range(4):
            start, stop = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            torch.cuda.synchronize()
            start.record()
            backend.dispatch(call, ws)
            stop.record()
            torch.cuda.synchronize()
            times.append(start.elapsed_time(stop))
        took.append(min(times))
    assert took[0] <= 2 * took[1], took


@pytest.mark.parametrize("m,past", [(300, 1537), (150, 4000)])
def test_bits_do_not_depend_on_capture_or_on_what_ran_before(torch_cuda, m, past):
    """One call: captured on a backend that has dispatched nothing, eager on a
    fresh one, and eager after a call that left a large scratch."""
    torch = torch_cuda
    b, h, hkv, d = 1, 32, 8, 128

    def made(m, past):
        g = torch.Generator(device="cuda")
        g.manual_seed(m + past)
        mk = lambda rows, heads: torch.randn((b * heads * rows, d), generator=g, device="cuda").to(torch.bfloat16)  # noqa: E731
        ops = [mk(m, h), mk(past, hkv), mk(past, hkv), mk(m, hkv), mk(m, hkv),
               torch.tensor([past], dtype=torch.int32, device="cuda"),
               torch.zeros((b * h * m, d), dtype=torch.bfloat16, device="cuda")]
        ws = DeviceWorkspace()
        for s, x in enumerate(ops):
            ws.bind(s, x)
        return ws, ops[-1], KernelCall.DecodeAttentionValid(DecodeAttentionValidCall(
            *[BufferRef(s) for s in range(7)], b, h, hkv, m, past, m, d, 0, DTYPE_BF16))

    ws, out, call = made(m, past)
    big_ws, _, big = made(1, 60000)
    got = []
    for how in ("captured", "eager", "after"):
        stream = torch.cuda.Stream()
        be = HipBackend(stream=stream.cuda_stream)
        torch.cuda.synchronize()
        out.zero_()
        torch.cuda.synchronize()
        if how == "captured":
            # (sizes that need scratch need it before a capture, as any call's do)
            if m < 256:
                be.dispatch(call, ws)
                be.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=stream):
                be.dispatch(call, ws)
            out.zero_()
            torch.cuda.synchronize()
            graph.replay()
        else:
            if how == "after":
                be.dispatch(big, big_ws)
            be.dispatch(call, ws)
        torch.cuda.synchronize()
        got.append(out.view(torch.int16).cpu())
        if how == "captured":
            del graph
        be.close()
    assert got[0].any()
    assert torch.equal(got[0], got[1]) and torch.equal(got[0], got[2])


@pytest.mark.parametrize("dtype", [DTYPE_BF16, DTYPE_F16])
@pytest.mark.parametrize("form", ["valid", "mask"])
@pytest.mark.parametrize("h,hkv,m,past,d", [
    (4, 1, 5, 30, 64),      # 20 rows: one slice and a quarter of the next
    (4, 1, 16, 100, 128),   # 64 rows of a tile
    (8, 2, 40, 70, 80),     # 160 rows: a tile and two of its slices
    (2, 2, 129, 200, 96),   # a tile and one row
])
def test_bits_do_not_depend_on_how_many_workgroups_share_a_tile(torch_cuda, backend, h, hkv, m, past, d, form, dtype):
    """A lone sequence's tiles are sliced among up to eight workgroups, those of 256
    sequences are not: every copy of the sequence has the lone one's bits."""
    rng, many = np.random.default_rng(m + d), 256
    make, wrap = ((DecodeAttentionCall, KernelCall.DecodeAttention) if form == "mask" else
                  (DecodeAttentionValidCall, KernelCall.DecodeAttentionValid))
    ops = [enc(rng.standard_normal(n * d), dtype) for n in (h * m, hkv * past, hkv * past, hkv * m, hkv * m)]
    last = ((rng.standard_normal((m, past + m)) * 2).astype(np.float32) if form == "mask" else
            np.array([past - 3], np.uint32))
    one = dispatch(torch_cuda, backend, make, wrap, ops, last.ravel(), (1, h, hkv, m, past, m, d), dtype)
    all_ = dispatch(torch_cuda, backend, make, wrap, [np.tile(x, many) for x in ops], last.ravel(),
                    (many, h, hkv, m, past, m, d), dtype)
    assert np.isfinite(one).all() and one.any()
    assert np.array_equal(np.tile(one, (many, 1, 1, 1)).view(np.uint32), all_.view(np.uint32))
