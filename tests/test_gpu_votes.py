"""The vote kernel at the edges of its pair chunks (128 pairs, masks padded with zeros) and of its fitness forms."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("values", [(-1, 0, 1), (-3, 2, 5)], ids=["ternary", "any"])
@pytest.mark.parametrize("pairs", [1, 127, 128, 129, 640])
def test_votes_and_update_at_chunk_edges(pkg, orc, dev, pairs, values):
    import torch
    kw = dict(hidden=64, head_dim=32, n_layers=3, seq_len=32, population=2 * pairs)
    ocfg = orc.config(**kw)
    ctx = pkg.Context(pkg.default_config(**kw))
    model = orc.init_model(ocfg, 42)
    state = np.zeros(model.size, orc.ADAM_DTYPE)
    ctx.model_upload(model)
    fit = np.random.default_rng(pairs).choice(np.array(values, np.int32), pairs)
    seed, lr = 0xFFFFFF00, 5.0                       # pair seeds that wrap around 2^32
    d_fit = torch.from_numpy(fit).to(dev)
    d_seed = torch.from_numpy(np.array([seed], np.uint32).view(np.int32)).to(dev)
    d_lr = torch.tensor([lr], dtype=torch.float32, device=dev)
    for t in (t for t in ctx.tensors() if t["is_matrix"]):
        d_votes = torch.zeros(t["rows"] * t["cols"], dtype=torch.int32, device=dev)
        ctx.matrix_votes(t["id"], d_fit.data_ptr(), d_seed.data_ptr(), d_votes.data_ptr())
        ctx.sync()
        ref = np.zeros(t["rows"] * t["cols"], np.int32)
        orc.lib().orc_matrix_votes(C.byref(ocfg), t["rows"], t["cols"], t["off_a"], t["off_b"], t["seed_base"],
                                   fit.ctypes.data_as(C.c_void_p), pairs, C.c_uint32(seed), ref.ctypes.data_as(C.c_void_p))
        assert np.array_equal(d_votes.cpu().numpy(), ref), t["name"]
    for _ in range(2):
        ctx.es_update(d_fit.data_ptr(), d_seed.data_ptr(), d_lr.data_ptr())
        n_ref = orc.es_update_adam(ocfg, model, state, fit, seed, lr)
        assert np.array_equal(ctx.model_download(), model)
        assert np.array_equal(ctx.opt_state_download().view(np.int32), state.view(np.int32))
        assert ctx.last_update_count() == n_ref
    ctx.close()


@pytest.mark.parametrize("values", [(-1, 0, 1), (-3, 2, 5)], ids=["ternary", "any"])
@pytest.mark.parametrize("pairs", [1, 129])
def test_update_in_wide_tiles(pkg, orc, dev, pairs, values):
    """The same in the 128 x 128 tiles that a model of this size takes."""
    import torch
    kw = dict(hidden=512, head_dim=32, n_layers=1, seq_len=32, population=2 * pairs)
    ocfg = orc.config(**kw)
    ctx = pkg.Context(pkg.default_config(**kw))
    model = orc.init_model(ocfg, 42)
    state = np.zeros(model.size, orc.ADAM_DTYPE)
    ctx.model_upload(model)
    fit = np.random.default_rng(pairs).choice(np.array(values, np.int32), pairs)
    seed, lr = 0x12345678, 5.0
    d_fit = torch.from_numpy(fit).to(dev)
    d_seed = torch.tensor([seed], dtype=torch.int32, device=dev)
    d_lr = torch.tensor([lr], dtype=torch.float32, device=dev)
    for _ in range(2):
        ctx.es_update(d_fit.data_ptr(), d_seed.data_ptr(), d_lr.data_ptr())
        n_ref = orc.es_update_adam(ocfg, model, state, fit, seed, lr)
        assert np.array_equal(ctx.model_download(), model)
        assert np.array_equal(ctx.opt_state_download().view(np.int32), state.view(np.int32))
        assert ctx.last_update_count() == n_ref
    ctx.close()


@pytest.mark.parametrize("pairs", [1, 129])
@pytest.mark.parametrize("hidden,vocab", [(64, 768), (128, 16384)], ids=["64_tiles", "128_tiles"])
def test_embedding_columns_behind_the_layers_rows(pkg, orc, dev, hidden, vocab, pairs):
    """The noise table's rows from 4 hidden on are shorter ones, for the columns of the embedding alone."""
    import torch
    kw = dict(hidden=hidden, head_dim=32, n_layers=2, seq_len=32, vocab=vocab, population=2 * pairs)
    ocfg = orc.config(**kw)
    ctx = pkg.Context(pkg.default_config(**kw))
    fit = np.random.default_rng(pairs).choice(np.array([-1, 1], np.int32), pairs)
    seed, d_fit = 0xFFFFFFF0, torch.from_numpy(fit).to(dev)
    d_seed = torch.from_numpy(np.array([seed], np.uint32).view(np.int32)).to(dev)
    t = next(t for t in ctx.tensors() if t["name"] == "embedding")
    ref = np.zeros(t["rows"] * t["cols"], np.int32)
    orc.lib().orc_matrix_votes(C.byref(ocfg), t["rows"], t["cols"], t["off_a"], t["off_b"], t["seed_base"],
                               fit.ctypes.data_as(C.c_void_p), pairs, C.c_uint32(seed), ref.ctypes.data_as(C.c_void_p))
    d_votes = torch.zeros(ref.size, dtype=torch.int32, device=dev)
    ctx.matrix_votes(t["id"], d_fit.data_ptr(), d_seed.data_ptr(), d_votes.data_ptr())
    ctx.sync()
    assert np.array_equal(d_votes.cpu().numpy(), ref)
    # and in the launch of a whole update: the first moment of an untouched state is (1 - beta1) * -vote
    d_lr = torch.zeros(1, dtype=torch.float32, device=dev)
    ctx.es_update(d_fit.data_ptr(), d_seed.data_ptr(), d_lr.data_ptr())
    at = ctx.tensor_state_offset(t["id"]) // 4
    m = ctx.opt_state_download()[at:at + 3 * ref.size:3]
    assert np.array_equal(m, (np.float32(1) - np.float32(ctx.cfg.adam_beta1)) * -ref.astype(np.float32))
    ctx.close()


@pytest.mark.parametrize("muon", [0, 1])
def test_timed_update_has_both_classes_and_the_same_results(pkg, dev, muon):
    import torch
    got = []
    for timed in (False, True):
        ctx = pkg.Context(pkg.default_config(hidden=64, head_dim=32, n_layers=2, seq_len=32, population=40, use_muon=muon))
        ctx.model_init(42)
        fit = torch.from_numpy(np.random.default_rng(1).integers(-1, 2, 20).astype(np.int32)).to(dev)
        seed, lr = torch.tensor([5], dtype=torch.int32, device=dev), torch.tensor([5.0], device=dev)
        ctx.enable_timing(timed)
        for _ in range(2):
            ctx.es_update(fit.data_ptr(), seed.data_ptr(), lr.data_ptr())
        got.append((ctx.model_download(), ctx.opt_state_download(), ctx.last_update_count()))
        if timed:
            launches = {k: v[0] for k, v in ctx.timing().items()}
            assert launches["update_vector"] == 2 and launches["update_matrix"] >= 2, launches
        ctx.close()
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1]) and got[0][2] == got[1][2] > 0
