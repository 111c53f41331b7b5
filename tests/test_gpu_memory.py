"""Device memory that a context takes, by the driver's figure around the calls."""
import pytest

pytestmark = pytest.mark.gpu


def _free(dev):
    import torch
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info(dev)[0]


def test_first_generation_takes_no_logits_of_the_whole_window(pkg, dev):
    """Logits of every position of the window (128 MiB here) are for the form without the K / V cache alone."""
    import torch
    warm = pkg.Context(pkg.default_config(hidden=64, head_dim=32, n_layers=1, seq_len=32, vocab=65536, population=2))
    b = torch.zeros(512, dtype=torch.int32, device=dev)
    warm.model_init(1)
    warm.generate(b.data_ptr(), 2, 4, 1)                 # the kernels' code is resident from here on
    warm.sync()
    ctx = pkg.Context(pkg.default_config(hidden=64, head_dim=32, n_layers=1, seq_len=512, vocab=65536, population=2))
    ctx.model_init(1)
    ctx.sync()
    before = _free(dev)
    ctx.generate(b.data_ptr(), 2, 4, 1)
    ctx.sync()
    assert before - _free(dev) < 32 << 20
    want = b.cpu()
    ctx.generate_kv_cache(False)
    ctx.generate(b.data_ptr(), 2, 4, 1)
    ctx.sync()
    assert before - _free(dev) >= 96 << 20 and torch.equal(b.cpu(), want)
    ctx.close()
    warm.close()


def test_context_of_a_large_vocabulary(pkg, dev):
    """The noise table takes the embedding's columns by their own windows (about 25 MB), not with every layer's seeds (0.5 GB)."""
    warm = pkg.Context(pkg.default_config(hidden=64, head_dim=32, n_layers=1, seq_len=32, population=2))
    before = _free(dev)
    ctx = pkg.Context(pkg.default_config(hidden=64, head_dim=32, n_layers=8, seq_len=32, vocab=65536, population=2))
    assert before - _free(dev) < 160 << 20               # 9 MB of weights, 54 MB of optimizer state, the table
    ctx.close()
    warm.close()
