"""The pair tile kernels where a tile of 128 positions runs on over the ends of
rows: one row per tile and less, rows one short of and one past a tile, and a
last tile that is nearly empty.  Every operator that writes the pair in place,
both orders of the rows, against the float64 CPU oracle (rms 1e-2, max 8e-2 of
the update, the bounds the operators have on any size)."""

import pytest
import torch

from oracle import af3_oracle as O

pytestmark = pytest.mark.gpu
D = torch.float64


def compare(name, got, want):
    got, want = got.double().cpu(), want.double()
    scale = float((want ** 2).mean().sqrt())
    rms, mx = float(((got - want) ** 2).mean().sqrt()) / scale, float((got - want).abs().max()) / scale
    print(f"{name}: rms {rms:.3e} max {mx:.3e}", flush=True)
    assert torch.isfinite(got).all() and rms <= 1e-2 and mx <= 8e-2, (name, rms, mx)


@pytest.mark.parametrize("n", [2, 5, 17, 63, 65, 127, 129])
def test_rows_that_end_inside_a_tile(gpu_pkg, n):
    g = torch.Generator().manual_seed(n)
    pair = O.round_bf16(torch.randn(n, n, 128, generator=g))
    mask = (torch.rand(n, n, generator=g) > 0.2).float()
    mask[:, 0] = 1
    for flag in (False, True):
        for make, cls, kw, ref in (
                (O.make_triangle_multiplication_params, "TriangleMultiplication", dict(_outgoing=flag),
                 lambda p: O.triangle_multiplication(pair.double(), mask.double(), p, flag)),
                (lambda g: O.make_grid_self_attention_params(g, std=0.1), "GridSelfAttention",
                 dict(num_head=4, transpose=flag),
                 lambda p: O.grid_self_attention(pair.double(), mask.double(), p, 4, flag))):
            params = {k: O.round_bf16(v) for k, v in make(g).items()}
            mod = getattr(gpu_pkg.nn, cls)(c_pair=128, **kw)
            mod.load_state_dict(params)
            mod.to("cuda:0")
            compare(f"{cls} n={n} {flag}", mod(pair.to("cuda:0"), mask.to("cuda:0")), ref(O.cast_params(params, D)))
