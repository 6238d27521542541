"""The triangle contraction at few tokens, on the kernel that takes a channel's panels in one trip and on either side of its line."""

import threading

import pytest
import torch

from oracle import af3_oracle as O

# One row, edges of 32-row blocks and of a row's 16-byte chunks, every tiling of 1 to 10 blocks, the last sizes and the first past them.
N_128 = [1, 7, 9, 31, 32, 33, 64, 65, 96, 97, 129, 161, 193, 207, 208, 209, 223, 224, 225]
N_64 = [1, 33, 100, 161, 200, 225, 256, 257, 288, 289, 303, 304, 305]


@pytest.mark.gpu
@pytest.mark.parametrize("n", N_128)
def test_panels(gpu_pkg, n):
    """fp32 sums of bf16 products, one rounding to bf16 (half a unit in 2^8, and the sums' order).

    The columns from n to ld are nobody's: the kernels leave different things there."""
    g = torch.Generator(device="cuda").manual_seed(n)
    ld = (n + 7) // 8 * 8
    a, b = (torch.zeros(128, n, ld, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    for x in (a, b):
        x[..., :n] = torch.randn(128, n, n, generator=g, device="cuda")
    got = gpu_pkg.ops.triangle_contraction(a, b, out=torch.full_like(a, float("nan")))
    want = torch.bmm(a.double(), b.double().transpose(1, 2).contiguous())
    assert ((got[..., :n].double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4 * n ** 0.5).all()


@pytest.mark.gpu
@pytest.mark.parametrize("n", N_64)
def test_panels_of_half_the_channels(gpu_pkg, n):
    """A triangle multiplication of 64 channels against the float64 oracle, to the update's tolerance at this width (rms 1e-2,
    largest error 8e-2 of the rms)."""
    g = torch.Generator().manual_seed(n)
    p = {k: O.round_bf16(v) for k, v in O.make_triangle_multiplication_params(g, 64, std=0.1).items()}
    pair = O.round_bf16(torch.randn(n, n, 64, generator=g)).cuda()
    mask = (torch.rand(n, n, generator=g) > 0.15).float().cuda()
    mod = gpu_pkg.nn.TriangleMultiplication(c_pair=64, _outgoing=True)
    mod.load_state_dict(p)
    got = mod.cuda()(pair, mask).double()
    want = O.triangle_multiplication(pair.double(), mask.double(), {k: v.double().cuda() for k, v in p.items()}, True)
    scale = want.pow(2).mean().sqrt()
    assert (got - want).pow(2).mean().sqrt() <= 1e-2 * scale and (got - want).abs().max() <= 8e-2 * scale


@pytest.mark.gpu
def test_panels_of_several_sizes_from_several_threads(gpu_pkg):
    """Sizes that ask for different amounts of LDS, launched by threads with a stream each."""
    g = torch.Generator(device="cuda").manual_seed(1)
    sizes, got, failed = (97, 160, 193, 224), {}, []
    start = threading.Barrier(len(sizes))
    ops = {n: [torch.randn(128, n, (n + 7) // 8 * 8, generator=g, device="cuda").bfloat16() for _ in range(2)] for n in sizes}
    for n in sizes:
        for x in ops[n]:
            x[..., n:] = 0
    want = {n: gpu_pkg.ops.triangle_contraction(*ops[n]) for n in sizes}
    torch.cuda.synchronize()

    def work(n):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                start.wait()
                got[n] = [gpu_pkg.ops.triangle_contraction(*ops[n]) for _ in range(100)]
                torch.cuda.current_stream().synchronize()
        except Exception as e:
            failed.append((n, e))
    threads = [threading.Thread(target=work, args=(n,)) for n in sizes]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed
    for n in sizes:
        assert all(torch.equal(x[..., :n], want[n][..., :n]) for x in got[n])
