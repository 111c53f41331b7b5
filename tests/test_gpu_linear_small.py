"""The one-launch linear layer for few rows against the kernels that rearrange W first: parts of a 128-column group, every depth, one
tile, members of several tiles, the largest call that takes it and the next one."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("noise", ["pair", "own", "none"])
@pytest.mark.parametrize("members,T,K,N", [(1, 32, 64, 64), (3, 64, 64, 256), (5, 32, 128, 128), (2, 64, 256, 64), (3, 128, 256, 448), (1, 64, 512, 192),
                                           (7, 64, 512, 384), (2, 32, 1024, 256), (1, 32, 512, 512), (64, 32, 256, 512), (64, 64, 512, 512), (65, 64, 512, 512)])
def test_small_linear_equals_the_streaming_kernels(pkg, dev, members, T, K, N, noise):
    import torch
    g = torch.Generator("cuda").manual_seed(K + N + members)
    ctx = pkg.Context(pkg.default_config(population=2, seq_len=32))
    x = torch.randint(-128, 128, (members * T, K), dtype=torch.int8, device=dev, generator=g)
    w = torch.randint(-128, 128, (K * N,), dtype=torch.int8, device=dev, generator=g)
    out = []
    for direct in (True, False):
        if not direct and (K, N) == (256, 512) and T % 64:
            continue                                            # no streaming instance
        ctx.linear_kernel(direct)
        y32 = torch.full((members * T, N), 7, dtype=torch.int32, device=dev)
        y8 = torch.full((members * T, N), 7, dtype=torch.int8, device=dev)
        only = torch.full((members * T, N), 7, dtype=torch.int8, device=dev)
        args = (x.data_ptr(), w.data_ptr(), members, T, K, N)
        for a, b in ((y32.data_ptr(), y8.data_ptr()), (None, only.data_ptr())):
            if noise == "none":
                ctx.shared_linear(*args, 8, a, b)
            else:
                (ctx.perturbed_linear if noise == "pair" else ctx.perturbed_linear_own_noise)(*args, 0xFFFFFFF0, 200, 201, 8, a, b)
        ctx.sync()
        assert torch.equal(y8.int(), y32.clamp(-127, 127)) and torch.equal(only, y8)
        out.append(y32)
    assert torch.equal(out[0], out[-1])
    ctx.close()
