"""The column slices that k_mlp and k_qkv take at larger populations (use_many_slices, use_one_slice_*), against the oracle: losses of
sampled members of chunks that are just large enough (more than stage taps hold), with windows that fill a workgroup's tiles, share it with other members, or need several passes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw,overlay", [
    (dict(hidden=256, head_dim=64, seq_len=32, population=1538), False),      # one slice in k_qkv only, four members to a workgroup
    (dict(hidden=256, head_dim=64, seq_len=64, population=770), False),       # two members, the last workgroup not full
    (dict(hidden=256, head_dim=32, seq_len=128, population=386), False),      # first block by value: two slices there
    (dict(hidden=256, head_dim=64, seq_len=256, population=194), False),
    (dict(hidden=256, head_dim=64, seq_len=512, population=98), False),
    (dict(hidden=256, head_dim=64, seq_len=128, population=386, vocab=512), False),         # first block at every position
    (dict(hidden=256, head_dim=64, seq_len=64, population=770, shift_mlp_down=23), False),  # accumulators that do not hold the residual
    (dict(hidden=256, head_dim=64, seq_len=64, population=770, shift_out=24), False),
    (dict(hidden=256, head_dim=64, seq_len=64, population=770, noise_mask=31, sigma_shift=5), False),
    (dict(hidden=256, head_dim=64, seq_len=64, population=770), True),
    (dict(hidden=128, head_dim=32, seq_len=64, population=514), False),       # few slices below hidden 256
    (dict(hidden=64, head_dim=32, seq_len=32, population=1026), False)],
    ids=["t32", "t64", "t128", "t256", "t512", "vocab", "down23", "out24", "wide_noise", "overlay", "h128", "h64"])
def test_slices_follow_the_oracle(pkg, orc, kw, overlay):
    import torch
    kw = dict(n_layers=2, **kw)
    P = kw["population"]
    members = sorted({0, 1, 2, 3, P // 3, P // 2, P - 4, P - 3, P - 2, P - 1})
    ocfg = orc.config(**kw)
    data = orc.zipf_bytes(1 << 18)
    if kw.get("vocab", 256) > 256:
        data = ((data[0::2].astype(np.uint32) << 8 | data[1::2]) % kw["vocab"]).astype(np.uint32)
    model = orc.init_model(ocfg, 42)
    rng = np.random.default_rng(7)
    for t in orc.tensor_table(ocfg):
        if not t["is_matrix"]:
            model[t["offset"]:t["offset"] + t["cols"]] += rng.integers(-9, 10, t["cols"]).astype(np.int8)
    ctx = pkg.Context(pkg.default_config(**kw))
    ctx.model_upload(model)
    ov = None
    if overlay:
        ov = rng.integers(-10, 90, model.size).astype(np.int8)
        ctx.adaptive_enable()
        ctx.overlay_upload(ov)
    d_data = torch.from_numpy(data.view(np.int32) if data.dtype == np.uint32 else data).cuda()
    loss = torch.zeros(P, dtype=torch.int32, device="cuda")
    ctx.population_forward(d_data.data_ptr(), len(data), 11, 4321, 0, P, loss.data_ptr())
    ctx.sync()
    got = loss.cpu().numpy()
    ref = [orc.forward_member(ocfg, model, data, 11, 4321, m, **({"overlay": ov} if overlay else {})) for m in members]
    assert [int(got[m]) for m in members] == [r[0] if isinstance(r, tuple) else r for r in ref]
    assert len(set(got.tolist())) > P // 8
    ctx.close()
