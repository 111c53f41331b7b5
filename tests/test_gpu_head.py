"""The head over more than 256 entries: logits that climb far above the first block's (the counters move), all logits equal (every
count in one place), tables that end too late for the counters, and windows of one to eight tiles."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["climbing", "equal", "random"])
@pytest.mark.parametrize("kw", [dict(hidden=64, seq_len=32, vocab=512, population=6), dict(hidden=128, seq_len=64, vocab=768, population=6),
                                dict(hidden=256, seq_len=128, vocab=2048, population=2), dict(hidden=512, seq_len=256, vocab=768, population=2),
                                dict(hidden=128, seq_len=32, vocab=1024, population=6, softmax_exp_scale=9.0),
                                dict(hidden=128, seq_len=32, vocab=1024, population=6, softmax_exp_scale=14.0)],
                         ids=["h64_t32", "h128_t64", "h256_t128", "h512_t256", "table_to_112", "table_to_175"])
def test_head_counts_follow_the_oracle(pkg, orc, dev, kw, kind):
    import torch
    kw = dict(kw, head_dim=32, n_layers=1)
    ocfg = orc.config(**kw)
    model = orc.init_model(ocfg, 42)
    ctx = pkg.Context(pkg.default_config(**kw))
    t = next(t for t in ctx.tensors() if t["name"] == "embedding")
    emb = model[t["offset"]:t["offset"] + t["rows"] * t["cols"]].reshape(t["rows"] // 4, t["cols"], 4)
    if kind == "climbing":                                     # weights grow along the vocabulary
        scale = np.linspace(0, 1, kw["vocab"])[None, :, None]
        emb[...] = np.random.default_rng(5).integers(-127, 128, emb.shape) * scale
    if kind == "equal":
        emb[...] = 0
    rng = np.random.default_rng(7)
    data = rng.integers(0, kw["vocab"], 4096).astype(np.uint32)
    ctx.model_upload(model)
    d_data = torch.from_numpy(data.view(np.int32)).to(dev)
    loss = torch.zeros(kw["population"], dtype=torch.int32, device=dev)
    ctx.population_forward(d_data.data_ptr(), len(data), 11, 987654321, 0, kw["population"], loss.data_ptr())
    ctx.sync()
    assert loss.cpu().tolist() == [orc.forward_member(ocfg, model, data, 11, 987654321, m) for m in range(kw["population"])]
    ctx.close()
