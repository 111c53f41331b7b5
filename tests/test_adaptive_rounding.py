"""The adaptive normalisation's rounding as one fused multiply-add: the identity on the CPU, and the forward on both sides of
the range in which it is used."""
import numpy as np
import pytest

LIMIT, MULTIPLES_FROM = 33157, 10414


def _reference(val, mx):
    """egg_adaptive_normalize.h:10-103 in float32: the product, then half away from zero"""
    s = np.float32(127.0) / (np.float32(mx) + np.float32(1e-9))
    p = (val.astype(np.float32) * s).astype(np.float64)
    return np.where(p >= 0, np.floor(p + 0.5), np.ceil(p - 0.5)).astype(np.int64)


def _fused(val, mx):
    """adaptive_fused_scale and the fused sum: the products of a whole number below 2^24 and a float32 are exact in float64"""
    s = np.float32(127.0) / (np.float32(mx) + np.float32(1e-9))
    tie = np.float32(np.float32(mx) * np.float32(0.5)) * s
    if tie >= np.float32(63.5) and np.float64(mx) * np.float64(s) - 127.0 <= 0.0:
        s = np.nextafter(s, np.float32(np.inf), dtype=np.float32)
    return np.rint(val.astype(np.float64) * np.float64(s)).astype(np.int64)


def test_fused_rounding_equals_the_reference():
    """Every value of every maximum in a sample that holds all multiples of 254, the ends of the range and 1,500 others."""
    rng = np.random.default_rng(3)
    maxima = set(range(1, 300)) | set(range(254, LIMIT, 254)) | set(range(LIMIT - 100, LIMIT)) | set(rng.integers(1, LIMIT, 1500).tolist())
    differ = set()
    for mx in sorted(maxima):
        val = np.arange(-mx, mx + 1)
        if not np.array_equal(_reference(val, mx), _fused(val, mx)):
            differ.add(mx)
    assert all(mx >= MULTIPLES_FROM and mx % 254 == 0 for mx in differ), sorted(differ)
    assert MULTIPLES_FROM in differ and len(differ) == 15


@pytest.mark.gpu
@pytest.mark.parametrize("hidden,head_dim,spread", [(64, 32, 127), (128, 32, 100), (256, 64, 46), (256, 64, 127), (512, 64, 32)])
def test_forward_on_both_sides_of_the_fused_range(pkg, orc, hidden, head_dim, spread):
    """Weights spread so that the row maxima in front of Q, K and V lie around or beyond the bound: every stage against the oracle."""
    import torch
    from oracle import forward_numpy as fn
    kw = dict(hidden=hidden, head_dim=head_dim, n_layers=1, seq_len=64, population=4)
    ocfg = orc.config(**kw)
    data = orc.zipf_bytes(1 << 14)
    model = orc.init_model(ocfg, 42)
    rng = np.random.default_rng(spread)
    for t in orc.tensor_table(ocfg):
        if t["is_matrix"]:
            sl = slice(t["offset"], t["offset"] + t["rows"] * t["cols"])
            model[sl] = rng.integers(-spread, spread + 1, t["rows"] * t["cols"]).astype(np.int8)
    maxima = []
    normalize = fn.adaptive_normalize
    fn.adaptive_normalize = lambda val: (maxima.append(np.abs(val).max(axis=1)), normalize(val))[1]
    try:
        fn.forward_member(ocfg, model, orc.tensor_table(ocfg), orc.tables(ocfg), data, 7, 99, 1)
    finally:
        fn.adaptive_normalize = normalize
    qkv = np.concatenate(maxima[1:4])
    assert qkv.max() >= LIMIT and np.concatenate(maxima).min() < LIMIT, (qkv.min(), qkv.max())
    ctx = pkg.Context(pkg.default_config(**kw))
    ctx.model_upload(model)
    ctx.enable_taps(True)
    d_data = torch.from_numpy(data).cuda()
    loss = torch.zeros(4, dtype=torch.int32, device="cuda")
    ctx.population_forward(d_data.data_ptr(), len(data), 7, 99, 0, 4, loss.data_ptr())
    ctx.sync()
    for m in range(4):
        ref_loss, tr = orc.forward_member(ocfg, model, data, 7, 99, m, trace=True)
        for st in ("q", "k", "v", "x_attn", "x_mlp"):
            assert np.array_equal(ctx.tap(f"{st}.0", m), tr[st][0]), (m, st)
        assert int(loss[m]) == ref_loss
    ctx.close()
