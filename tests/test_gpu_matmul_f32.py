"""GPU parity of the f32 MatMul, row-major and panel-packed B, at the edges of
each of its forms (64 x 64 tiles; K split over a workgroup's waves, 32 x 32,
32 x 16 and 16 x 16; the general one): ragged rows, columns and k, operands
aligned to 4 bytes only. The form a shape takes is worked out from the launcher's
own table and asserted. (Row-major B, up to 64 rows, k a multiple of 16 and n of
4, aligned: the few-row kernel of its own.)

Bound: a sum of k products rounded to f32 at each step, in any order, is within
k 2^-24 of the sum of the products' magnitudes (to first order); compared
element by element against the f64 product. Beyond the operands' last elements
memory holds NaN and around the output a pattern, so a read past an edge or a
store past one shows; an Inf at the end of one row of A and a NaN in one column
of B stay in that row / column."""
import re
from pathlib import Path

import pytest

import hologram_amd
from hologram_amd import DTYPE_F32, BufferRef, DeviceWorkspace, KernelCall, MatMulCall

pytestmark = pytest.mark.gpu
GUARD = 1024


def taken(m, k, n):
    """launch_matmul_f32's choice, on the model in its source: (rows, columns) of a
    workgroup's tile, None for the general kernel."""
    if max(k, n) >= 1 << 22:
        return None
    source = (Path(hologram_amd.__file__).parent / "csrc" / "gemm_f32.hip").read_text()
    table = re.search(r"F32Form kF32Forms\[\] = \{(.*?)\n\};", source, re.S).group(1)
    forms = re.findall(r"\{(\d+), (\d+), (\d+), \d+, ([\d.]+)f\}", table)
    assert len(forms) == 4

    def time(f):
        tm, tn, step = map(int, f[:3])
        tiles = -(-m // tm) * -(-n // tn)
        return float(f[3]) * (-(-k // step) * step) * ((tiles + 255) // 256)

    best = min(forms, key=time)
    return int(best[0]), int(best[1])


def guarded(torch, values, fill, offset):
    whole = torch.full((values.numel() + 2 * GUARD,), fill, dtype=torch.float32, device="cuda")
    lo = GUARD + offset
    whole[lo:lo + values.numel()] = values.reshape(-1)
    return whole, whole[lo:lo + values.numel()]


def run(torch, backend, m, k, n, packed, poison=False, offset=0, whole=False):
    g = torch.Generator(device="cuda")
    g.manual_seed(m + k + n)
    if whole:   # -1, 0 or 1
        a = torch.randint(-1, 2, (m, k), generator=g, device="cuda").float()
        b = torch.randint(-1, 2, (k, n), generator=g, device="cuda").float()
    else:
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


# form -> m, k, n
SHAPES = {
    (16, 16): [(1, 2048, 4096), (7, 1000, 333), (16, 515, 40), (65, 2000, 260)],
    (32, 16): [(50, 1024, 2048), (50, 1023, 2047), (45, 1531, 2001), (300, 700, 300)],
    (32, 32): [(200, 2047, 1021), (33, 700, 4003)],
    (64, 64): [(1, 1, 1), (17, 64, 100), (255, 3, 257), (500, 160, 2000), (449, 129, 2049), (1000, 130, 1001),
               (513, 31, 1984), (1024, 256, 1024), (2049, 97, 130)],
}
CASES = [(form, *mkn) for form, some in SHAPES.items() for mkn in some]


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("form,m,k,n", CASES)
def test_f32_edges(torch_cuda, backend, form, m, k, n, packed):
    assert taken(m, k, n) == form
    for offset in (0, 1):
        got, a, b = run(torch_cuda, backend, m, k, n, packed, offset=offset)
        want = a.double() @ b.double()
        bound = (a.abs().double() @ b.abs().double()) * (k * 2.0 ** -24)
        assert bool(((got.double() - want).abs() <= bound + 1e-30).all()), offset


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("form,m,k,n", [((16, 16), 33, 1021, 77), ((16, 16), 8, 999, 4096),
                                        ((32, 16), 45, 1531, 2001), ((32, 32), 200, 2046, 1021),
                                        ((64, 64), 500, 1543, 2001)])
def test_f32_non_finite_stays_in_its_row_and_column(torch_cuda, backend, form, m, k, n, packed):
    assert taken(m, k, n) == form
    got, _, _ = run(torch_cuda, backend, m, k, n, packed, poison=True)
    torch = torch_cuda
    bad = ~torch.isfinite(got)
    rows, cols = torch.zeros(m, dtype=bool, device="cuda"), torch.zeros(n, dtype=bool, device="cuda")
    rows[m // 2], cols[n // 2] = True, True
    assert torch.equal(bad, rows[:, None] | cols[None, :])


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("m,k,n", [(1, (1 << 22) + 3, 5), (130, 2, (1 << 22) + 5)])
def test_f32_general_kernel(torch_cuda, backend, m, k, n, packed):
    """k or n past the other forms' 32-bit ranges. Whole numbers whose sums stay
    below 2^24 in any order: equal to the last bit."""
    assert taken(m, k, n) is None and k < 1 << 24
    got, a, b = run(torch_cuda, backend, m, k, n, packed, offset=1, whole=True)
    for r in range(0, m, 43):
        assert torch_cuda.equal(got[r].double(), (a[r].double()[:, None] * b.double()).sum(0))
