"""GPU parity of the f32 MatMul, row-major and panel-packed B, at the edges of
each of its forms (64 x 64 tiles; K split over a workgroup's waves, 32 x 32,
32 x 16 and 16 x 16): ragged rows, columns and k, operands aligned to 4 bytes only.

Bound: a sum of k products rounded to f32 at each step, in any order, is within
k 2^-24 of the sum of the products' magnitudes (to first order); compared
element by element against the f64 product. Beyond the operands' last elements
memory holds NaN and around the output a pattern, so a read past an edge or a
store past one shows; an Inf at the end of one row of A and a NaN in one column
of B stay in that row / column."""
import pytest

from hologram_amd import DTYPE_F32, BufferRef, DeviceWorkspace, KernelCall, MatMulCall

pytestmark = pytest.mark.gpu
GUARD = 1024


def guarded(torch, values, fill, offset):
    whole = torch.full((values.numel() + 2 * GUARD,), fill, dtype=torch.float32, device="cuda")
    lo = GUARD + offset
    whole[lo:lo + values.numel()] = values.reshape(-1)
    return whole, whole[lo:lo + values.numel()]


def run(torch, backend, m, k, n, packed, poison=False, offset=0):
    g = torch.Generator(device="cuda")
    g.manual_seed(m + k + n)
    a = torch.randn((m, k), generator=g, device="cuda")
    b = torch.randn((k, n), generator=g, device="cuda")
    if poison:
        a[m // 2, k - 1] = float("inf")
        b[0, n // 2] = float("nan")
    p = b
    if packed:
        p = torch.zeros((k, (n + 15) // 16 * 16), device="cuda")
        p[:, :n] = b
        p = p.view(k, -1, 16).permute(1, 0, 2).contiguous()
    wa, va = guarded(torch, a, float("nan"), offset)
    wb, vb = guarded(torch, p, float("nan"), offset)
    wo, vo = guarded(torch, torch.zeros(m * n, device="cuda"), 7.0, offset)
    ws = DeviceWorkspace()
    for s, v in enumerate((va, vb, vo)):
        ws.bind(s, ptr=v.data_ptr(), nbytes=v.numel() * 4)
    backend.dispatch(KernelCall.MatMul(MatMulCall(BufferRef(0), BufferRef(1), BufferRef(2), m, k, n, DTYPE_F32,
                                                  b_packed=packed)), ws)
    backend.synchronize()
    lo = GUARD + offset
    assert bool((wo[:lo] == 7.0).all()) and bool((wo[lo + m * n:] == 7.0).all())
    return vo.view(m, n), a, b


SHAPES = [  # m, k, n
    (1, 1, 1), (1, 2048, 4096), (7, 1000, 333), (16, 515, 40), (17, 64, 100),       # 16 x 16, 32 x 16
    (50, 1024, 2048), (65, 2000, 260), (200, 2047, 1021), (255, 3, 257),            # 32 x 16, 32 x 32
    (500, 160, 2000), (449, 129, 2049), (1000, 130, 1001), (513, 31, 1984),         # 64 x 64
    (1024, 256, 1024), (2049, 97, 130),
]


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("m,k,n", SHAPES)
def test_f32_edges(torch_cuda, backend, m, k, n, packed):
    for offset in (0, 1):
        got, a, b = run(torch_cuda, backend, m, k, n, packed, offset=offset)
        want = a.double() @ b.double()
        bound = (a.abs().double() @ b.abs().double()) * (k * 2.0 ** -24)
        assert bool(((got.double() - want).abs() <= bound + 1e-30).all()), offset


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("m,k,n", [(33, 1021, 77), (8, 999, 4096), (200, 2046, 1021), (500, 1543, 2001)])
def test_f32_non_finite_stays_in_its_row_and_column(torch_cuda, backend, m, k, n, packed):
    got, _, _ = run(torch_cuda, backend, m, k, n, packed, poison=True)
    torch = torch_cuda
    bad = ~torch.isfinite(got)
    rows, cols = torch.zeros(m, dtype=bool, device="cuda"), torch.zeros(n, dtype=bool, device="cuda")
    rows[m // 2], cols[n // 2] = True, True
    assert torch.equal(bad, rows[:, None] | cols[None, :])
