"""A model's blocks in one launch (k_blocks) against the same stages launched one by one (which a context that times its stages takes) and, for sampled members, against
the oracle: short windows, all hidden sizes that take it, both head widths, full and partial last workgroups, few and many column slices, and populations on both sides of the line."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [
    dict(hidden=64, head_dim=32, seq_len=32, population=64, n_layers=2),
    dict(hidden=64, head_dim=64, seq_len=32, population=2, n_layers=1),
    dict(hidden=64, head_dim=32, seq_len=64, population=1022, n_layers=2),           # 511 workgroups
    dict(hidden=64, head_dim=64, seq_len=64, population=1026, n_layers=1),           # 513: stage by stage
    dict(hidden=64, head_dim=64, seq_len=32, population=2042, n_layers=2),           # the last workgroup holds two of four members
    dict(hidden=128, head_dim=32, seq_len=64, population=1002, n_layers=3),
    dict(hidden=128, head_dim=64, seq_len=64, population=10, n_layers=5),
    dict(hidden=128, head_dim=64, seq_len=64, population=1024, n_layers=1),
    dict(hidden=128, head_dim=32, seq_len=32, population=1030, n_layers=2),
    dict(hidden=128, head_dim=64, seq_len=32, population=6, n_layers=2, vocab=512),
    dict(hidden=256, head_dim=64, seq_len=32, population=6, n_layers=2),
    dict(hidden=64, head_dim=64, seq_len=128, population=130, n_layers=2),
    dict(hidden=64, head_dim=32, seq_len=128, population=512, n_layers=1),
    dict(hidden=128, head_dim=64, seq_len=128, population=66, n_layers=2),
    dict(hidden=128, head_dim=32, seq_len=128, population=514, n_layers=1),         # stage by stage
    dict(hidden=256, head_dim=64, seq_len=128, population=130, n_layers=2),
    dict(hidden=256, head_dim=32, seq_len=128, population=302, n_layers=1),
    dict(hidden=256, head_dim=32, seq_len=64, population=250, n_layers=2),          # two passes: the first block once per byte value
    dict(hidden=256, head_dim=64, seq_len=64, population=512, n_layers=1),
    dict(hidden=256, head_dim=64, seq_len=64, population=514, n_layers=1),
    dict(hidden=256, head_dim=64, seq_len=32, population=1002, n_layers=2),
    dict(hidden=256, head_dim=64, seq_len=64, population=770, n_layers=1),          # one column slice: stage by stage
    dict(hidden=128, head_dim=32, seq_len=32, population=130, n_layers=2, noise_mask=31),     # noise that the launch does not take
    dict(hidden=64, head_dim=32, seq_len=32, population=130, n_layers=2, use_same_data=1)],
    ids=lambda kw: "h%(hidden)d_d%(head_dim)d_t%(seq_len)d_p%(population)d" % kw)
def test_blocks_equal_the_stages(pkg, orc, kw):
    import torch
    P, rng = kw["population"], np.random.default_rng(3)
    ocfg = orc.config(**kw)
    data = orc.zipf_bytes(1 << 17)
    if kw.get("vocab", 256) > 256:
        data = ((data[0::2].astype(np.uint32) << 8 | data[1::2]) % kw["vocab"]).astype(np.uint32)
    model = orc.init_model(ocfg, 42)
    for t in orc.tensor_table(ocfg):
        if not t["is_matrix"]:
            model[t["offset"]:t["offset"] + t["cols"]] += rng.integers(-9, 10, t["cols"]).astype(np.int8)
    ctx = pkg.Context(pkg.default_config(**kw))
    ctx.model_upload(model)
    d_data = torch.from_numpy(data.view(np.int32) if data.dtype == np.uint32 else data).cuda()

    def losses(seed, first=0, count=P):
        out = torch.zeros(count, dtype=torch.int32, device="cuda")
        ctx.population_forward(d_data.data_ptr(), len(data), 11, seed, first, count, out.data_ptr())
        ctx.sync()
        return out.cpu().numpy()

    def stages(seed, *part):
        ctx.enable_timing(True, stages=True)
        got = losses(seed, *part)
        ctx.enable_timing(False)
        return got
    for seed in (4321, 5):                              # a second step through the same buffers
        got = losses(seed)
        assert np.array_equal(got, stages(seed))
        members = sorted({0, 1, P // 2, P - 2, P - 1})
        ref = [orc.forward_member(ocfg, model, data, 11, seed, m) for m in members]
        assert [int(got[m]) for m in members] == [r[0] if isinstance(r, tuple) else r for r in ref]
    if P > 4:                                           # a worker's part of the population
        assert np.array_equal(losses(4321, 2, P - 3), stages(4321, 2, P - 3))
    ctx.close()


@pytest.mark.parametrize("overlay", [False, True])
def test_timing_describes_the_launches_of_an_untimed_forward(pkg, orc, overlay):
    import torch
    layers = 3
    ctx = pkg.Context(pkg.default_config(hidden=128, head_dim=32, seq_len=64, population=66, n_layers=layers))
    ctx.model_init(42)
    if overlay:                                         # the launch for all blocks does not take it
        ctx.adaptive_enable()
    data = torch.from_numpy(orc.zipf_bytes(1 << 14)).cuda()
    loss = torch.zeros(66, dtype=torch.int32, device="cuda")
    for stages in (False, True, False):
        ctx.enable_timing(True, stages=stages)
        ctx.timing_reset()
        for seed in (1, 2):
            ctx.population_forward(data.data_ptr(), data.numel(), 0, seed, 0, 66, loss.data_ptr())
        got = {k: v[0] for k, v in ctx.timing().items() if v[0]}
        one = not stages and not overlay
        assert got == ({"blocks": 2, "head": 2} if one else {"mlp_first": 2, "qkv": 2 * layers, "attn": 2 * layers, "mlp": 2 * layers, "head": 2}), got
        assert all(ms > 0 for n, ms in ctx.timing().values() if n)
    ctx.close()
