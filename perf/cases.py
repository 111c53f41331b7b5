"""The work that programs of this framework have it do, as measurable cases.

Six kinds of pass, each through the public entry points as a user's program calls them:

  step      one ES step of the transformer (forward of the population, fitness, votes, AdamW), eager or as the captured
            graph, with or without the adaptive noise overlay, then what the training loop reads back of it
  worker    a d-eggs worker's part of a step: the forward of its range of the population, the losses on the host, the
            shaped fitness and its base-3 packing for the wire
  update    votes and optimizer step from a fitness vector that came from elsewhere (AdamW or Muon), and the new weights
            (with `checkpoint`: the optimizer state too) on the host
  generate  a sampled continuation of a prompt, with the plain or the d-eggs sampler
  gru       one step of the full_trained_egg.c program (recurrent forward of the population, threshold update)
  linear    one perturbed (or shared-weight) int8 linear layer over a population's activations
"""
import math

import numpy as np
import torch

from __graft_entry__ import load_package

pkg = load_package()

STREAM = 1 << 22          # tokens of a synthetic stream


# --------------------------------------------------------------------------------------------------------------- cases
def step(hidden, head_dim, layers, seq, population, graph=False, overlay=False):
    return dict(kind="step", hidden=hidden, head_dim=head_dim, layers=layers, seq=seq, population=population, graph=graph, overlay=overlay)


def worker(hidden, head_dim, layers, seq, vocab, first, count):
    return dict(kind="worker", hidden=hidden, head_dim=head_dim, layers=layers, seq=seq, vocab=vocab, first=first, count=count)


def update(hidden, head_dim, layers, population, muon, checkpoint):
    return dict(kind="update", hidden=hidden, head_dim=head_dim, layers=layers, population=population, muon=muon, checkpoint=checkpoint)


def generate(hidden, head_dim, layers, seq, vocab, prompt, new, deggs):
    return dict(kind="generate", hidden=hidden, head_dim=head_dim, layers=layers, seq=seq, vocab=vocab, prompt=prompt, new=new, deggs=deggs)


def gru(hidden, layers, seq, population):
    return dict(kind="gru", hidden=hidden, layers=layers, seq=seq, population=population)


def linear(members, tokens, k, n, noise, out):
    return dict(kind="linear", members=members, tokens=tokens, k=k, n=n, noise=noise, out=out)


def listed():
    return [
        # a first experiment on a toy model: the call is launches and latency
        dict(step(64, 32, 2, 32, 64), name="step_toy"),
        # a sweep of small models over short windows, the step captured once; the population fills no tile or block evenly
        dict(step(128, 32, 3, 64, 1002, graph=True), name="step_small_graph"),
        # the benchmark's training step
        dict(step(256, 64, 4, 256, 40960), name="step_40960"),
        # the same model trained with d-eggs' adaptive noise overlay
        dict(step(256, 64, 4, 256, 2048, overlay=True), name="step_overlay"),
        # a worker of a distributed d-eggs run on its chunk, byte vocabulary
        dict(worker(512, 64, 8, 512, 256, 4096, 2048), name="worker_d_eggs"),
        # a worker with d-eggs' default vocabulary and a ragged range
        dict(worker(512, 64, 8, 256, 8192, 1026, 510), name="worker_vocab_8192"),
        # a coordinator's update of a small model with the checkpoint that it keeps
        dict(update(128, 32, 4, 8192, False, True), name="update_checkpoint"),
        # the Muon update of the d-eggs-style model
        dict(update(512, 64, 8, 16384, True, False), name="update_muon"),
        # the sample that the training loop prints: 32 tokens continued by 64
        dict(generate(256, 64, 4, 256, 256, 32, 64, False), name="generate_bytes"),
        # d-eggs' sampler on its vocabulary
        dict(generate(512, 64, 8, 256, 8192, 32, 64, True), name="generate_d_eggs"),
        # full_trained_egg.c at its defaults
        dict(gru(512, 4, 4096, 128), name="gru_4096"),
        # one layer over a large population's activations
        dict(linear(8192, 128, 512, 512, "pair", "int8"), name="linear_8192"),
    ]


def spread(rng, lo, hi, unit=1):
    """a multiple of `unit` from [lo, hi], even in its logarithm"""
    return max(lo, min(hi, unit * round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / unit)))


MOST_OPS = 6e13           # of one drawn pass: about three quarters of the largest listed one


def draw(rng):
    kind = rng.choice(["step", "step", "worker", "update", "generate", "gru", "linear"])
    hidden = rng.choice([64, 128, 256, 512])
    head_dim = rng.choice([32, 64])
    if kind == "step":
        c = step(hidden, head_dim, rng.randint(1, 6), rng.choice([32, 64, 128, 256]), spread(rng, 64, 40960, 2), rng.random() < 0.4)
        c["overlay"] = not c["graph"] and rng.random() < 0.3
        most = MOST_OPS / (3 if c["overlay"] else 1)         # the overlay's sums are taken term by term
        c["population"] = max(2, min(c["population"], 2 * int(c["population"] / 2 * most / forward_ops(c))))
        return c
    if kind == "worker":
        c = worker(rng.choice([256, 512]), 64, rng.randint(2, 8), rng.choice([128, 256, 512]), 256 * rng.choice([1, 1, 2, 3, 8, 32]),
                   2 * rng.randint(0, 4096), spread(rng, 64, 4096, 2))
        c["count"] = max(2, min(c["count"], 2 * int(c["count"] / 2 * MOST_OPS / forward_ops(c))))
        return c
    if kind == "update":
        muon = rng.random() < 0.5
        return update(hidden, head_dim, rng.randint(1, 8), spread(rng, 64, 16384, 2), muon, not muon and hidden <= 128)
    if kind == "generate":
        deggs = rng.random() < 0.5
        seq = rng.choice([64, 128, 256, 512])
        prompt = rng.randint(1, min(hidden, seq // 2))
        new = rng.randint(8, min(96, (min(seq, 256) if deggs else seq) - min(prompt, 128)))
        prompt = min(prompt, 128)
        vocab = 256 * rng.choice([1, 1, 3, 8, 32])
        return generate(hidden, head_dim, rng.randint(1, 8), seq, vocab, prompt, new if vocab <= 2048 else min(new, 40), deggs)
    if kind == "gru":
        return gru(hidden, rng.randint(1, 4), spread(rng, 64, 4096), rng.choice([32, 64, 96, 128]))
    k = rng.choice([256, 512])
    return linear(spread(rng, 1, 8192), 64 * rng.randint(1, 2), k, 64 * rng.randint(1, 8), rng.choice(["pair", "own", "none"]), rng.choice(["int8", "int32"]))


# ------------------------------------------------------------------------------------------------------------- work
def forward_ops(c):
    """int8 operations of the shared products of one forward: 12 H^2 weights a layer, 8 H^2 in front, attention, the head"""
    h, members = c["hidden"], c.get("population", c.get("count", 1))
    token = 2 * (12 * h * h * c["layers"] + 8 * h * h + c["layers"] * h * (c["seq"] + 1) + h * c.get("vocab", 256))
    return token * members * c["seq"]


def params(c):
    h = c["hidden"]
    return 12 * h * h * c["layers"] + 8 * h * h + h * c.get("vocab", 256)


def work(case):
    c, kind = case, case["kind"]
    if kind == "linear":
        rows = c["members"] * c["tokens"]
        return {"bytes": rows * (c["k"] + c["n"] * (4 if c["out"] == "int32" else 1)) + c["k"] * c["n"], "flops": 2 * rows * c["k"] * c["n"]}
    if kind == "gru":
        h, token = c["hidden"], c["population"] * c["seq"]
        weights = c["layers"] * 12 * h * h + 256 * h
        return {"bytes": 3 * weights + 2 * c["population"] * c["layers"] * h + token, "flops": 2 * token * weights + c["population"] * weights}
    if kind == "generate":
        return {"bytes": params(c) + 8 * (c["prompt"] + c["new"]), "flops": 2 * params(c) * (c["prompt"] + c["new"])}
    if kind == "worker":
        return {"bytes": params(c) + c["count"] * (4 + c["seq"]), "flops": forward_ops(c)}
    votes = params(c) * c["population"]                       # a multiplication and an addition for each pair
    state = params(c) * (2 + (16 if c.get("muon") else 24))   # weights and optimizer state, in and out
    if kind == "update":
        out = params(c) * (13 if c["checkpoint"] else 1)      # and what goes to the host
        ns = 20 * 6 * c["hidden"] ** 3 * c["layers"] if c["muon"] else 0
        return {"bytes": state + out + 2 * c["population"], "flops": votes + ns}
    return {"bytes": state + c["population"] * (8 + c["seq"]), "flops": forward_ops(c) + votes}


def tolerance(case):
    # Integers throughout, and AdamW is a fixed sequence of IEEE operations.  Muon's float32 matrix products have no fixed
    # order: a weight whose accumulator comes to lie within rounding of a threshold may differ.
    return {"rel": 1e-5, "differ": 1e-3} if case["kind"] == "update" and case["muon"] else "exact"


# ------------------------------------------------------------------------------------------------------------- state
class State:
    pass


def generator(seed):
    g = torch.Generator("cuda")
    g.manual_seed(seed)
    return g


def stream_of(g, vocab):
    """Zipf(1.1) bytes over a permutation of the byte values; larger vocabularies: uint32 tokens from pairs of them"""
    n = STREAM if vocab == 256 else 2 * STREAM
    weights = 1.0 / torch.arange(1, 257, device="cuda", dtype=torch.float64) ** 1.1
    rank = torch.searchsorted(torch.cumsum(weights / weights.sum(), 0), torch.rand(n, device="cuda", generator=g, dtype=torch.float64))
    data = torch.randperm(256, device="cuda", generator=g)[rank.clamp_(max=255)]
    if vocab == 256:
        return data.to(torch.uint8)
    return ((data[0::2] * 256 + data[1::2]) % vocab).to(torch.int32)


def training_state(g, cfg):
    """Optimizer state of a run under way: moments of the size that the votes of this population have, accumulators
    anywhere between their thresholds (so every update moves some weights)."""
    tensors, _, size = pkg.describe_layout(cfg)
    vote = 75.0 * math.sqrt(cfg.population / 2)
    state = torch.empty(size // 4, device="cuda")
    for t in tensors:
        n, at, muon = t["rows"] * t["cols"], t["state_offset"] // 4, cfg.use_muon and t["muon"]
        s = state[at:at + n * (2 if muon else 3)].view(n, -1)
        s[:, 0].normal_(0.0, vote * (1.9 if muon else 0.23), generator=g)
        s[:, -1].uniform_(-1.0, 1.0, generator=g)
        if not muon:
            s[:, 1].uniform_(0.5 * vote * vote, vote * vote, generator=g)
    return state.cpu().numpy()


def prepare(case, seed):
    s = State()
    s.case, s.seed, s.passes = case, 1 + seed % 1000003, 0
    kind, g = case["kind"], generator(seed)
    if kind == "linear":
        rows = case["members"] * case["tokens"]
        s.x = torch.randint(-127, 128, (rows, case["k"]), dtype=torch.int8, device="cuda", generator=g)
        s.w = torch.randint(-127, 128, (case["k"] * case["n"],), dtype=torch.int8, device="cuda", generator=g)
        s.y = torch.empty((rows, case["n"]), dtype=torch.int32 if case["out"] == "int32" else torch.int8, device="cuda")
        s.ctx = pkg.Context(pkg.default_config(population=2, seq_len=32))
        return s
    if kind == "gru":
        s.data = stream_of(g, 256)
        s.ctx = pkg.GruContext(pkg.gru_default_config(hidden=case["hidden"], n_layers=case["layers"], seq_len=case["seq"], population=case["population"]))
        s.ctx.model_init(s.seed)
        s.ctx.state_reset()
        return s
    more = {"seq_len": case.get("seq", 32), "vocab": case.get("vocab", 256), "population": case.get("population", 2)}
    if kind == "worker":
        more.update(population=case["first"] + case["count"] + case["first"] % 4, chunk_members=case["count"])
    if kind == "update":
        more.update(chunk_members=2, use_muon=int(case["muon"]))
    cfg = pkg.default_config(hidden=case["hidden"], head_dim=case["head_dim"], n_layers=case["layers"], **more)
    s.ctx = pkg.Context(cfg)
    s.ctx.model_init(s.seed)
    if kind in ("step", "update"):
        s.ctx.opt_state_upload(training_state(g, cfg))
    if kind == "update":
        s.fit = torch.randint(-1, 2, (case["population"] // 2,), dtype=torch.int32, device="cuda", generator=g)
        s.step_seed = torch.tensor([s.seed], dtype=torch.int32, device="cuda")
        s.lr = torch.tensor([pkg.learning_rate(0)], device="cuda")
        return s
    if kind == "generate":
        s.buffer = torch.zeros(case["seq"], dtype=torch.uint8 if case["vocab"] == 256 else torch.int32, device="cuda")
        s.buffer[:case["prompt"]] = stream_of(g, case["vocab"])[:case["prompt"]]
        return s
    s.data = stream_of(g, cfg.vocab)
    if kind == "worker":
        s.loss = torch.zeros(cfg.population, dtype=torch.int32, device="cuda")
        return s
    if case["overlay"]:
        s.ctx.adaptive_enable()
        s.ctx.overlay_upload(torch.randint(16, 96, (s.ctx.model_bytes(),), dtype=torch.int8, device="cuda", generator=g).cpu().numpy())
    if case["graph"]:
        torch.cuda.synchronize()
        s.ctx.step_capture(s.data.data_ptr(), s.data.numel())
    return s


def run(s):
    c, ctx, k = s.case, s.ctx, s.passes
    s.passes += 1
    kind = c["kind"]
    if kind == "linear":
        args = (s.x.data_ptr(), s.w.data_ptr(), c["members"], c["tokens"], c["k"], c["n"])
        y32, y8 = (s.y.data_ptr(), None) if c["out"] == "int32" else (None, s.y.data_ptr())
        if c["noise"] == "none":
            ctx.shared_linear(*args, 8, y32, y8)
        elif c["noise"] == "own":
            ctx.perturbed_linear_own_noise(*args, s.seed, 200, 201, 8, y32, y8)
        else:
            ctx.perturbed_linear(*args, s.seed, 200, 201, 8, y32, y8)
        return s.y
    if kind == "generate":
        if c["deggs"]:
            ctx.generate_deggs(s.buffer.data_ptr(), c["prompt"], c["new"], s.seed + k)
        else:
            ctx.generate(s.buffer.data_ptr(), c["prompt"], c["new"], s.seed + k)
        return s.buffer
    if kind == "update":
        ctx.es_update(s.fit.data_ptr(), s.step_seed.data_ptr(), s.lr.data_ptr())
        out = {"model": ctx.model_download()}
        if c["checkpoint"]:
            out["state"] = ctx.opt_state_download()
        return out
    start = k * c["seq"] % (STREAM - c["seq"])
    if kind == "gru":
        ctx.step(s.data.data_ptr(), s.data.numel(), start, s.seed + k)
        loss, fit = ctx.losses()
        return {"loss": loss, "fit": fit, "recurrent": ctx.state_download(), "model": ctx.model_download()}
    if kind == "worker":
        ctx.population_forward(s.data.data_ptr(), s.data.numel(), start, s.seed + k, c["first"], c["count"], s.loss.data_ptr())
        ctx.sync()
        loss = s.loss[c["first"]:c["first"] + c["count"]].cpu().numpy()
        fit, total = pkg.shape_fitness(loss)
        return {"loss": loss, "fit": fit, "total": total, "wire": pkg.ternary_pack(fit)}
    if c["graph"]:
        ctx.step_launch(start, s.seed + k, pkg.learning_rate(0))
    else:
        ctx.step(s.data.data_ptr(), s.data.numel(), start, s.seed + k, pkg.learning_rate(0))
    out = {"updates": ctx.last_update_count()}
    out["loss"], out["fit"] = ctx.step_losses()
    out["model"] = ctx.model_download()        # the training loop takes the weights along where it prints a sample or saves
    if c["overlay"]:
        out["overlay"] = ctx.overlay_download()
    return out
