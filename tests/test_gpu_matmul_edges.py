"""GPU parity of the 16-bit tiled MatMul where its tiles end: rows, columns and
k that are no multiple of any tile or slab, in bf16 and f16, at sizes that take
each tile (256 x 256, 256 x 128, 128 x 128, 64 x 64) with and without ragged
edges; the residual form; a SwiGLU-shaped pair of ragged rows through a session.
The tile a shape takes is worked out from the launcher's own table and asserted,
so that a change of its costs cannot leave a tile untested.

Bounds. Against the f64 product of the same operands, normalized by the largest
result. A bf16 truncation loses less than one ulp, 2^-7 of the value; the
residual form truncates twice, the product (at most the largest product, here
below the largest sum) and the sum: 2^-6. f16 rounds, 2^-11 each time: 2^-10.
The f32 sums add at most k 2^-24, below 2^-11 of that. Beyond the operands' last elements memory holds NaN and the
output's surroundings a pattern, so a read past an edge or a store past one
shows; an Inf in one row of A and one column of B stays in that row / column."""
import re
from pathlib import Path

import numpy as np
import pytest

import hologram_amd

from hologram_amd import (DTYPE_BF16, DTYPE_F16, BufferRef, DeviceWorkspace, KernelCall, MatMulAddCall,
                          MatMulCall)

pytestmark = pytest.mark.gpu
GUARD = 4096


def taken(m, n):
    """best_tile of the launcher for one product, on the costs in its source."""
    source = (Path(hologram_amd.__file__).parent / "csrc" / "gemm.hip").read_text()
    table = re.search(r"TileCost kTiles\[4\] = \{(.*?)\};", source, re.S).group(1)
    tiles = [[float(x) for x in t] for t in re.findall(r"\{(\d+), (\d+), ([\d.]+)f, ([\d.]+)f\}", table)]
    assert len(tiles) == 4

    def cost(t):
        count = -(-m // int(t[0])) * -(-n // int(t[1]))
        rounds = (count + 255) // 256
        return (rounds - 1) * t[3] + t[2] + (t[3] - t[2]) * (count - (rounds - 1) * 256) / 256

    best = min(tiles, key=cost)
    return int(best[0]), int(best[1])


def whole_tiles(m, k, n):
    """No edge: whole tiles, and slabs in whole rounds of the stages."""
    bm, bn = taken(m, n)
    return m % bm == 0 and n % bn == 0 and (k % 64 == 0 if bm == 64 else k % 128 == 0 and k >= 256)


def guarded(torch, values, dtype, fill):
    """values followed (and preceded) by GUARD elements of `fill`; returns (whole, view)."""
    flat = values.reshape(-1).to(dtype)
    whole = torch.full((flat.numel() + 2 * GUARD,), fill, dtype=dtype, device="cuda")
    whole[GUARD:GUARD + flat.numel()] = flat
    return whole, whole[GUARD:GUARD + flat.numel()]


def run(torch, backend, m, k, n, dtype, residual, poison, seed):
    dt = torch.bfloat16 if dtype == DTYPE_BF16 else torch.float16
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    a = torch.randn((m, k), generator=g, device="cuda").to(dt)
    b = (torch.randn((k, n), generator=g, device="cuda") * k ** -0.5).to(dt)
    r = torch.randn((m, n), generator=g, device="cuda").to(dt)
    if poison:
        a[m // 2, k - 1] = float("inf")
        b[k - 1, n // 2] = float("nan")
    want = a.double() @ b.double()
    keep, ws = [], DeviceWorkspace()
    for s, x in enumerate((a, b, r)):
        whole, view = guarded(torch, x, dt, float("nan"))
        keep.append(whole)
        ws.bind(s, ptr=view.data_ptr(), nbytes=view.numel() * 2)
    whole, out = guarded(torch, torch.zeros(m, n, device="cuda"), dt, 7.0)
    ws.bind(3, ptr=out.data_ptr(), nbytes=out.numel() * 2)
    mm = MatMulCall(BufferRef(0), BufferRef(1), BufferRef(3), m, k, n, dtype)
    backend.dispatch(KernelCall.MatMulAdd(MatMulAddCall(mm, BufferRef(2))) if residual
                     else KernelCall.MatMul(mm), ws)
    backend.synchronize()
    assert bool((whole[:GUARD] == 7.0).all()) and bool((whole[GUARD + m * n:] == 7.0).all())
    return out.view(m, n).double(), want + r.double() if residual else want


# tile -> m, k, n with edges and without (bf16 of up to 64 rows: the few-row
# kernel, where its k and n allow)
SHAPES = {
    (64, 64): ([(1, 64, 4096), (65, 8, 136), (100, 200, 72), (63, 1000, 328), (333, 520, 1032), (700, 1096, 2056)],
               [(64, 512, 512), (512, 512, 512), (1024, 256, 2048)]),
    (128, 128): ([(1009, 264, 4096), (1009, 2048, 4088), (1500, 392, 2568)],
                 [(2048, 256, 2048), (1024, 384, 4096)]),
    (256, 128): ([(1009, 136, 4104), (2300, 264, 1800), (2047, 392, 8200)], [(2048, 256, 4096)]),
    (256, 256): ([(4097, 128, 2568), (2047, 136, 8184)], [(4096, 256, 4096), (2048, 384, 8192)]),
}
CASES = [(tile, edge, *mkn) for tile, (ragged, whole) in SHAPES.items()
         for edge, some in ((True, ragged), (False, whole)) for mkn in some]


@pytest.mark.parametrize("dtype", [DTYPE_BF16, DTYPE_F16])
@pytest.mark.parametrize("residual", [False, True])
@pytest.mark.parametrize("tile,edge,m,k,n", CASES)
def test_tile_edges(torch_cuda, backend, tile, edge, m, k, n, residual, dtype):
    assert taken(m, n) == tile and whole_tiles(m, k, n) == (not edge)
    got, want = run(torch_cuda, backend, m, k, n, dtype, residual, False, m + k + n)
    tol = 2.0 ** (-10 if dtype == DTYPE_F16 else -6 if residual else -7)
    assert float((got - want).abs().max() / want.abs().max()) <= tol


@pytest.mark.parametrize("dtype", [DTYPE_BF16, DTYPE_F16])
@pytest.mark.parametrize("tile,m,k,n", [((64, 64), 100, 200, 72), ((64, 64), 333, 520, 1032),
                                        ((128, 128), 1009, 264, 4096), ((128, 128), 1500, 392, 2568),
                                        ((256, 128), 1009, 136, 4104), ((256, 128), 2047, 392, 8200),
                                        ((256, 256), 2047, 136, 8184)])
def test_non_finite_operands_stay_in_their_row_and_column(torch_cuda, backend, tile, m, k, n, dtype):
    assert taken(m, n) == tile
    got, want = run(torch_cuda, backend, m, k, n, dtype, False, True, m + k + n)
    bad = ~torch_cuda.isfinite(got)
    expect = torch_cuda.zeros_like(bad)
    expect[m // 2, :] = True
    expect[:, n // 2] = True
    assert bool((bad == expect).all())
    tol = 2.0 ** (-7 if dtype == DTYPE_BF16 else -10)
    fine = ~expect
    assert float((got[fine] - want[fine]).abs().max() / want[fine].abs().max()) <= tol


@pytest.mark.parametrize("rows,ffn", [(67, 520), (100, 1032)])
def test_ragged_prompt_walk_fused_equals_unfused(torch_cuda, backend, rows, ffn):
    """q/k/v as one ragged launch, the SwiGLU pair and the residual adds in the
    tiled kernel's store: bit for bit the unfused walk."""
    from hologram_amd import HipSession
    from hologram_amd.decoder_graph import DecoderConfig, build_prefill, init_weights
    from hologram_amd.session import NO_DEVICE_FUSION
    from test_gpu_prefill import prefill_inputs, zero_caches
    cfg = DecoderConfig(layers=1, hidden=256, heads=4, kv_heads=2, head_dim=64, ffn=ffn, vocab=1000,
                        batch=3, bucket=128)
    archive = build_prefill(cfg, init_weights(cfg, seed=8, std=0.05), rows)
    prompt = np.random.default_rng(9).integers(0, cfg.vocab, (cfg.batch, rows))
    outs, nodes = [], []
    for flags in (0, NO_DEVICE_FUSION):
        s = HipSession(backend, archive, flags=flags)
        zero_caches(s.write_input, cfg)
        for i, b in enumerate(prefill_inputs(cfg, rows, prompt)):
            s.write_input(i, b)
        s.run()
        s.synchronize()
        outs.append([s.read_output(i) for i in range(len(s.outputs))])
        nodes.append(s.n_nodes)
        s.close()
    assert nodes[0] < nodes[1] - 3
    assert outs[0] == outs[1]
