"""Downloads of a context's memory: what was uploaded comes back, at sizes on both sides of each way of moving it (one piece,
pieces through the pinned slots, helpers and slots used again)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,layers,vocab", [(64, 1, 256), (128, 1, 256), (128, 4, 256), (256, 4, 768), (512, 8, 256)])
def test_download_returns_what_was_uploaded(pkg, hidden, layers, vocab):
    ctx = pkg.Context(pkg.default_config(hidden=hidden, head_dim=32, n_layers=layers, seq_len=32, vocab=vocab, population=2))
    rng = np.random.default_rng(hidden + layers)
    for _ in range(2):                                        # the second time through used slots
        model = rng.integers(-127, 128, ctx.model_bytes(), dtype=np.int8)
        state = rng.standard_normal(ctx.opt_state_download().size).astype(np.float32)
        ctx.model_upload(model)
        ctx.opt_state_upload(state)
        assert np.array_equal(ctx.model_download(), model)
        assert np.array_equal(ctx.opt_state_download(), state)
