"""The persistent decode launch against whole-window evaluation of every token (itself compared with the oracle in
test_gpu_parity.py): prompts and continuations around the blocks of 64 and 256 positions, every hidden size and head
width, vocabularies with fewer and more tiles than workgroups, two contexts at once, and captured replays."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(64, 32, 2, 64, 256, [(1, 1), (1, 63), (33, 31)]), (64, 64, 1, 512, 256, [(60, 10), (250, 12), (500, 12)]),
          (128, 32, 2, 256, 768, [(2, 5), (63, 3), (129, 70)]), (256, 64, 2, 256, 256, [(64, 2), (65, 66), (240, 16)]),
          (512, 64, 1, 512, 8192, [(1, 4), (190, 8), (317, 4)]), (64, 32, 1, 32, 65536, [(5, 6)])]


def _context(pkg, dev, hidden, head_dim, layers, seq, vocab):
    ctx = pkg.Context(pkg.default_config(hidden=hidden, head_dim=head_dim, n_layers=layers, seq_len=seq, vocab=vocab, population=2))
    ctx.model_init(42)
    model, rng = ctx.model_download(), np.random.default_rng(9)
    for t in ctx.tensors():
        n = t["rows"] * t["cols"]
        if t["name"] == "embedding":                     # a small tied head keeps the next-token distribution broad
            model[t["offset"]:t["offset"] + n] = rng.integers(-4, 5, n)
        elif not t["is_matrix"] and "bias" in t["name"]:
            model[t["offset"]:t["offset"] + n] = rng.integers(-20, 21, n)
    ctx.model_upload(model)
    return ctx


def _prompt(dev, vocab, n, total):
    import torch
    b = torch.zeros(total, dtype=torch.uint8 if vocab == 256 else torch.int32, device=dev)
    b[:n] = torch.from_numpy(np.random.default_rng(n).integers(0, vocab, n)).to(b.dtype).to(dev)
    return b


@pytest.mark.parametrize("deggs", [False, True], ids=["plain", "deggs"])
@pytest.mark.parametrize("hidden,head_dim,layers,seq,vocab,lengths", SHAPES, ids=["h%d_v%d_t%d" % (s[0], s[4], s[3]) for s in SHAPES])
def test_decode_equals_whole_window_evaluation(pkg, dev, hidden, head_dim, layers, seq, vocab, lengths, deggs):
    ctx = _context(pkg, dev, hidden, head_dim, layers, seq, vocab)
    seen = set()
    for n, new in lengths:
        if deggs and (n + new > 256 or n > hidden):
            continue
        got = []
        for cached in (True, False):
            ctx.generate_kv_cache(cached)
            b = _prompt(dev, vocab, n, n + new)
            (ctx.generate_deggs if deggs else ctx.generate)(b.data_ptr(), n, new, 1041)
            ctx.sync()
            got.append(b.cpu().numpy())
        assert np.array_equal(got[0], got[1]), (n, new, np.nonzero(got[0] != got[1])[0][:4])
        seen |= set(got[0][n:].tolist())
    assert len(seen) > 3 or not lengths
    ctx.close()


@pytest.mark.parametrize("hidden,head_dim", [(64, 32), (128, 64), (256, 64)])
def test_decode_with_the_largest_partial_sums(pkg, dev, hidden, head_dim):
    """Up to hidden 256 a strip's 64 intermediate and 16 attention values travel as partial sums of 21 bits.  Saturated
    intermediates (bias and weights at the ends of int8) on matrices of -128 and 127 make the largest ones there are,
    64 * 127 * 128, of both signs and in both halves of a message; two of every three columns stay random."""
    ctx = _context(pkg, dev, hidden, head_dim, 2, 128, 256)
    model, rng = ctx.model_download(), np.random.default_rng(3)
    names = set()
    for t in ctx.tensors():
        n = t["rows"] * t["cols"]
        if t["is_matrix"] and t["name"].startswith(("w_down", "w_o", "w_emb_mlp_down")):
            names.add(t["name"])
            block = model[t["offset"]:t["offset"] + n].reshape(-1, t["cols"], 4)      # four rows of a column together
            block[:, ::6], block[:, 3::6] = -128, 127
        elif not t["is_matrix"] and "up" in t["name"] and "bias" in t["name"]:
            model[t["offset"]:t["offset"] + n] = rng.choice(np.array([-128, 127], np.int8), n, p=[0.1, 0.9])
    ctx.model_upload(model)
    got = []
    for cached in (True, False):
        ctx.generate_kv_cache(cached)
        b = _prompt(dev, 256, 20, 84)
        ctx.generate(b.data_ptr(), 20, 64, 11)
        ctx.sync()
        got.append(b.cpu().numpy())
    assert len(names) == 5 and np.array_equal(got[0], got[1])
    ctx.close()


def test_decode_on_two_streams_and_replayed(pkg, dev):
    import torch
    ctxs = [_context(pkg, dev, h, 64, 2, 128, 256) for h in (256, 512)]
    want, bufs = [], []
    for ctx in ctxs:
        b = _prompt(dev, 256, 20, 80)
        ctx.generate(b.data_ptr(), 20, 60, 5)
        ctx.sync()
        want.append(b.cpu().numpy())
        bufs.append(_prompt(dev, 256, 20, 80))
    torch.cuda.synchronize()
    for _ in range(4):
        for ctx, b in zip(ctxs, bufs):
            ctx.generate(b.data_ptr(), 20, 60, 5)
    for ctx, b, w in zip(ctxs, bufs, want):
        ctx.sync()
        assert np.array_equal(b.cpu().numpy(), w)
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    ctxs[0].set_stream(stream.cuda_stream)
    with torch.cuda.graph(graph, stream=stream):
        ctxs[0].generate(bufs[0].data_ptr(), 20, 60, 5)
    for _ in range(3):
        bufs[0][20:] = 0
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(bufs[0].cpu().numpy(), want[0])
        bufs[0][20:] = 0
        torch.cuda.synchronize()
        ctxs[0].generate(bufs[0].data_ptr(), 20, 60, 5)          # eager between the replays
        ctxs[0].sync()
        assert np.array_equal(bufs[0].cpu().numpy(), want[0])
    for ctx in ctxs:
        ctx.close()


@pytest.mark.parametrize("hidden,head_dim,layers,seq,vocab,lengths", SHAPES, ids=["h%d_v%d_t%d" % (s[0], s[4], s[3]) for s in SHAPES])
def test_unanswered_waits_cost_time_only(pkg, dev, hidden, head_dim, layers, seq, vocab, lengths):
    """Waits that run into their bound (here: at once, or after a few polls, somewhere in the middle) leave the continuation
    to one workgroup: the tokens are the same in stream order, and the launches queued behind it are not disturbed."""
    ctx = _context(pkg, dev, hidden, head_dim, layers, seq, vocab)
    for n, new in lengths[-2:]:
        for generate in (ctx.generate, ctx.generate_deggs):
            if generate == ctx.generate_deggs and (n + new > 256 or n > hidden):
                continue
            bufs = [_prompt(dev, vocab, n, n + new) for _ in range(6)]
            for b, limit in zip(bufs, (1 << 23, 0, 1 << 23, 3, 20, 1 << 23)):
                ctx.generate_wait_limit(limit)
                generate(b.data_ptr(), n, new, 77)
            ctx.model_download()                         # any call that waits for the stream, no error
            got = [b.cpu().numpy() for b in bufs]
            assert all(np.array_equal(g, got[0]) for g in got), (n, new)
    ctx.close()
