"""What a user of the framework runs, as measurable cases: the Pairformer stack, the template embedding's 64-channel
blocks, the Evoformer (MSA) block, a whole trunk pass, and the diffusion head evaluated once, on a fresh batch, and
inside the sampling loop.  Inference only: the framework has no backward direction.

`listed()` are fixed points of those paths, `draw()` makes more of the same ranges, `prepare()` builds what a program
holds before the call (module with packed weights, batch, activations), `run()` is one pass through the public
modules, `work()` the arithmetic and traffic a pass cannot avoid, `tolerance()` how far two correct implementations
of the same precision may lie apart.
"""

from __future__ import annotations

import math

import torch

import __graft_entry__

af3 = __graft_entry__.load_package()

NOISE_LEVELS = 200       # steps of a sampling run: the conditioning is prepared for all of their noise levels
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}


def listed():
    return [
        # a short peptide: every kernel is tiny, launches and host work are what a user waits for
        dict(name="pairformer_n64", path="pairformer", n=64, blocks=4, dtype="bf16", padding=0),
        # the 4-block fp32-stream stack of the baseline configurations
        dict(name="pairformer_n128_f32", path="pairformer", n=128, blocks=4, dtype="f32", padding=0),
        # a domain-sized chain whose length fits no tile, a few padding tokens behind it
        dict(name="pairformer_n387", path="pairformer", n=387, blocks=4, dtype="bf16", padding=29),
        # the headline size, 10 % trailing padding
        dict(name="pairformer_n768", path="pairformer", n=768, blocks=4, dtype="bf16", padding=77),
        # the largest trunk size of the baseline configurations, nothing masked
        dict(name="pairformer_n1536", path="pairformer", n=1536, blocks=4, dtype="bf16", padding=0),
        # the template embedding's two blocks (64 channels, transition factor 2, no single track), ragged
        dict(name="template_n301", path="template", n=301, blocks=2, dtype="bf16", padding=11),
        # an MSA block at the MSA depth the trunk truncates to
        dict(name="evoformer_r1024_n768", path="evoformer", n=768, rows=1024, dtype="bf16", padding=77),
        # a shallow MSA over an odd token count: neither axis a multiple of anything
        dict(name="evoformer_r301_n187", path="evoformer", n=187, rows=301, dtype="bf16", padding=0),
        # a recycling pass of the trunk, 4 MSA blocks and 8 of the 48 Pairformer blocks (the others cost the same)
        dict(name="trunk_r128_n160", path="trunk", n=160, rows=128, padding=9),
        # one denoising evaluation on a prepared batch: what the sampler runs 200 times
        dict(name="denoise_n768", path="denoise", n=768, samples=5, padding=76),
        # a new batch: conditioning for all noise levels, per-batch state and the first evaluation
        dict(name="new_batch_n384", path="new_batch", n=384, samples=5, padding=20),
        # a sampling run on a small complex: many short evaluations one after the other
        dict(name="sampler_n100", path="sampler", n=100, samples=5, padding=4, steps=50),
    ]


def _log_between(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choices(["pairformer", "template", "evoformer", "trunk", "denoise", "new_batch", "sampler"],
                       [5, 1, 2, 1, 1, 1, 1])[0]
    pad = rng.choice([0.0, rng.uniform(0.0, 0.15)])
    if path == "pairformer":
        dtype = rng.choice(["bf16", "bf16", "bf16", "f32"])
        n = _log_between(rng, 40, 1536 if dtype == "bf16" else 1024)
        return dict(path=path, n=n, blocks=rng.randint(1, 4), dtype=dtype, padding=int(pad * n))
    if path == "template":
        n = _log_between(rng, 40, 768)
        return dict(path=path, n=n, blocks=2, dtype=rng.choice(["bf16", "f32"]), padding=int(pad * n))
    if path == "evoformer":
        n = _log_between(rng, 40, 768)
        return dict(path=path, n=n, rows=_log_between(rng, 16, 1024), dtype="bf16", padding=int(pad * n))
    if path == "trunk":
        n = _log_between(rng, 40, 384)
        return dict(path=path, n=n, rows=_log_between(rng, 16, 512), padding=int(pad * n))
    # the atom layout wants a token count that is a multiple of 4 (24 atom slots each, subsets of 32 atoms)
    n = 4 * _log_between(rng, 10, 64 if path == "sampler" else 192)
    case = dict(path=path, n=n, samples=rng.randint(1, 5), padding=int(pad * n))
    if path == "sampler":
        case["steps"] = rng.randint(20, 50)
    return case


# ------------------------------------------------------------------ inputs

def _module(make, gen, std):
    """A module on the GPU with random-init weights (matrices and biases N(0, std), LayerNorm weights around 1),
    packed for the kernels."""
    with torch.device("cuda"):
        mod = make()
    with torch.no_grad():
        for name, p in mod.named_parameters():
            p.normal_(0.0, std, generator=gen)
            if p.dim() == 1 and name.endswith("weight"):
                p += 1.0
    mod.invalidate()
    return mod.load_hip_params()


def _masks(n, padding):
    seq = (torch.arange(n, device="cuda") < n - padding).float()
    return seq, (seq[:, None] * seq[None, :]).contiguous()


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    host_gen = torch.Generator().manual_seed(seed)
    nn, path, n, padding = af3.nn, case["path"], case["n"], case["padding"]

    def normal(*shape):
        return torch.randn(*shape, generator=gen, device="cuda")

    st = dict(path=path)
    if path in ("pairformer", "template", "evoformer"):
        dtype = DTYPES[case["dtype"]]
        st["seq_mask"], st["pair_mask"] = _masks(n, padding)
        if path == "pairformer":
            st["mod"] = _module(lambda: nn.PairformerStack(num_blocks=case["blocks"]), gen, 0.02)
            st["pair"], st["single"] = normal(n, n, 128).to(dtype), normal(n, 384).to(dtype)
        elif path == "template":
            st["mods"] = [_module(lambda: nn.PairformerBlock(c_pair=64, num_intermediate_factor=2, with_single=False),
                                  gen, 0.02) for _ in range(case["blocks"])]
            st["pair"] = normal(n, n, 64).to(dtype)
        else:
            st["mod"] = _module(nn.EvoformerBlock, gen, 0.02)
            st["pair"], st["msa"] = normal(n, n, 128).to(dtype), normal(case["rows"], n, 64).to(dtype)
            cover = (torch.rand(case["rows"], n, generator=gen, device="cuda") > 0.2).float()
            cover[0] = 1.0                                   # the query sequence itself has no gaps
            st["msa_mask"] = (cover * st["seq_mask"]).contiguous()
        return st
    if path == "trunk":
        st["mod"] = _module(lambda: nn.Evoformer(pairformer_num_layer=8), gen, 0.02)
        st["batch"] = nn.atom_layout.synthetic_trunk_batch(n, case["rows"], host_gen, padding).to("cuda")
        st["target_feat"] = normal(n, 447)
        st["prev"] = {"pair": normal(n, n, 128), "single": normal(n, 384)}      # of the previous recycling pass
        return st
    head = st["mod"] = _module(nn.DiffusionHead, gen, 0.05)
    batch = st["batch"] = nn.atom_layout.synthetic_batch(n, host_gen, n_padding_tokens=padding).to("cuda")
    emb = st["emb"] = {"single": normal(n, 384), "pair": normal(n, n, 128), "target_feat": normal(n, 447)}
    steps = case.get("steps", NOISE_LEVELS)
    sampler = nn.DiffusionSampler(head, num_samples=case["samples"], diffusion_steps=steps)
    if path == "sampler":
        st["sampler"] = sampler
        st["positions"] = normal(case["samples"], n, 24, 3)
        st["rotations"] = torch.linalg.qr(torch.randn(steps, 3, 3, generator=host_gen))[0].to("cuda")
        st["translations"] = normal(steps, 3)
        return st
    st["t_hat"] = sampler.schedule(torch.device("cuda"))[1]
    st["step"] = steps // 2                              # a noise level in the middle of the schedule
    st["positions"] = normal(case["samples"], n, 24, 3) * float(st["t_hat"][st["step"]])
    if path == "denoise":
        st["single_cond"], st["pair_cond"] = head.pre_conditioning(batch, emb, st["t_hat"], True)
        st["state"] = head.prepare(batch, emb, st["pair_cond"])
    return st


# ------------------------------------------------------------------ one pass

@torch.no_grad()
def run(st):
    path = st["path"]
    if path == "pairformer":
        # the stack updates its tensors in place: it gets a copy, as a program keeps what it built them from
        return st["mod"](st["pair"].clone(), st["pair_mask"], st["single"].clone(), st["seq_mask"])
    if path == "template":
        pair = st["pair"].clone()
        for blk in st["mods"]:
            pair = blk(pair, st["pair_mask"])
        return pair
    if path == "evoformer":
        return st["mod"](st["msa"].clone(), st["pair"].clone(), st["msa_mask"], st["pair_mask"])
    if path == "trunk":
        out = st["mod"](st["batch"], st["prev"], st["target_feat"])
        return out["pair"], out["single"]
    if path == "sampler":
        return st["sampler"](st["batch"], st["emb"], positions=st["positions"], rotations=st["rotations"],
                             translations=st["translations"])["atom_positions"]
    head, batch, emb, t = st["mod"], st["batch"], st["emb"], st["t_hat"]
    i = st["step"]
    if path == "denoise":
        return head(st["positions"], t[i], batch, emb, st["single_cond"][i], st["pair_cond"], state=st["state"])
    single_cond, pair_cond = head.pre_conditioning(batch, emb, t, True)
    state = head.prepare(batch, emb, pair_cond)
    x = head(st["positions"], t[i], batch, emb, single_cond[i], pair_cond, state=state)
    return single_cond, pair_cond, x


# ------------------------------------------------------------------ what a pass cannot do without

def _pair_ops_flops(n, c, heads, factor):
    """Triangle multiplication and attention, both directions, and the pair transition on [n, n, c]."""
    trimul = 2 * c * n ** 3 + 12 * c * c * n ** 2
    triattn = 4 * c * n ** 3 + (10 * c * c + 2 * c * heads) * n ** 2
    return 2 * trimul + 2 * triattn + 6 * factor * c * c * n ** 2


def _pairformer_flops(n):
    single = 2 * 128 * 16 * n ** 2 + 4 * 384 * n ** 2 + 34 * 384 * 384 * n       # logits, attention, products
    return _pair_ops_flops(n, 128, 4, 4) + single


def _evoformer_flops(n, rows):
    outer = 2 * (32 * n) ** 2 * rows + 2 * n * n * 1024 * 128 + 2 * rows * n * 64 * 64
    average = 2 * 64 * rows * n * n + 6 * rows * n * 64 * 64 + 2 * 128 * 8 * n * n
    return outer + average + 24 * 64 * 64 * rows * n + _pair_ops_flops(n, 128, 4, 4)


def _denoise_flops(n, samples):
    rows, atoms = samples * n, samples * n * 12.5                # 1 to 24 atoms per token, evenly spread
    token = 24 * (2 * rows * 768 * 11 * 768 + 4 * rows * n * 768) + 2 * n * 384 * 24 * 6 * 768
    atom = 6 * (2 * atoms * 128 * 11 * 128 + 4 * atoms * 128 * 128) + 2 * atoms * 128 * 768 + 2 * rows * 768 * 128
    return token + atom


def _setup_flops(n, levels):
    pair = 2 * n * n * 128 * (267 + 2 * 768 + 24 * 16)           # first layer, two transitions, all pair logits
    return pair + 2 * levels * n * 384 * 2 * 2304 + 2 * n * 831 * 384


def work(case):
    path, n = case["path"], case["n"]
    item = 2 if case.get("dtype") == "bf16" else 4
    pair128 = 128 * n * n
    block_weights = 2 * (36 * 128 * 128 + 17 * 384 * 384)
    if path == "pairformer":
        b = 2 * item * (pair128 + 384 * n) + 4 * n * n + case["blocks"] * block_weights
        return {"bytes": b, "flops": case["blocks"] * _pairformer_flops(n)}
    if path == "template":
        return {"bytes": 2 * item * 64 * n * n + 4 * n * n, "flops": case["blocks"] * _pair_ops_flops(n, 64, 4, 2)}
    if path == "evoformer":
        rows = case["rows"]
        b = 2 * item * (pair128 + 64 * rows * n) + 4 * (n * n + rows * n)
        return {"bytes": b, "flops": _evoformer_flops(n, rows)}
    if path == "trunk":
        rows = case["rows"]
        b = 4 * (pair128 + 384 * n) + 2 * (pair128 + 384 * n) + 4 * 35 * rows * n + 8 * block_weights
        return {"bytes": b, "flops": 4 * _evoformer_flops(n, rows) + 8 * _pairformer_flops(n)}
    samples = case["samples"]
    weights = 2 * (24 * (11 * 768 * 768 + 6 * 384 * 768) + 6 * 11 * 128 * 128)
    positions = 2 * 4 * samples * n * 24 * 3
    if path == "denoise":
        return {"bytes": 4 * pair128 + weights + positions, "flops": _denoise_flops(n, samples)}
    levels = case.get("steps", NOISE_LEVELS)
    b = 2 * 4 * pair128 + 4 * levels * n * 384 + weights
    if path == "new_batch":
        return {"bytes": b + positions, "flops": _setup_flops(n, levels) + _denoise_flops(n, samples)}
    return {"bytes": b + levels * (4 * pair128 + weights + positions),
            "flops": _setup_flops(n, levels) + levels * _denoise_flops(n, samples)}


def tolerance(case):
    # bf16 products throughout.  On a bf16 residual stream every operator rounds the stream itself (0.2 % rms each);
    # on an fp32 stream only the updates carry bf16 error.  The sampler chains its evaluations.
    if case["path"] == "sampler":
        return {"rel": 2e-2, "max": 0.3}
    if case.get("dtype") == "f32":
        return {"rel": 5e-3, "max": 0.1}
    return {"rel": 1e-2, "max": 0.2}
