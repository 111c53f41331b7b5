"""The Newton-Schulz products on bf16 parts of float32 operands, against the iteration in 64 bits: one to many chunks of k, odd numbers of
them, both tile sizes, both operand orders, and the shapes next to the kernel's (sides that are not multiples of 64)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [(64, 64), (64, 96), (96, 64), (64, 160), (224, 64), (64, 448), (128, 128), (192, 128), (128, 544),
                                       (256, 256), (256, 1024), (512, 512), (512, 2048), (2048, 512)])
@pytest.mark.parametrize("scale", [1e-3, 140.0])
def test_iteration_against_64_bits(pkg, rows, cols, scale):
    import torch
    ctx = pkg.Context(pkg.default_config(hidden=512, head_dim=64, n_layers=1, seq_len=32, population=2, use_muon=1))
    g = torch.Generator().manual_seed(rows * 7 + cols)
    x = torch.randn(rows, cols, generator=g) * scale
    y = x.double() / x.double().norm()
    short = min(rows, cols)
    eye = 3.0 * torch.eye(short, dtype=torch.float64)
    for _ in range(5):
        y = 0.5 * ((eye - y @ y.T) @ y) if rows < cols else 0.5 * (y @ (eye - y.T @ y))
    d = x.cuda()
    ctx.newton_schulz(d.data_ptr(), rows, cols, 5)
    ctx.sync()
    err = float((d.cpu().double() - y).norm() / y.norm())
    # measured: at most 2.8e-7 (512 x 512); 6.0e-7 there with one accumulator through every bf16 instruction, 9.1e-7 with the float32 instruction
    assert err < 4.5e-7, err
    ctx.close()


def hard_pairs(n, seed):
    """float32 pairs in [1, 2) whose bf16 parts x = x0 + x1 + x2 have the largest x1 y2 + x2 y1 + x2 y2 of many: up to half a unit of the product's last place"""
    rng = np.random.default_rng(seed)

    def parts(x):
        out, left = [], x.copy()
        for _ in range(3):
            u = left.view(np.uint32)
            p = ((u + 0x7fff + ((u >> 16) & 1)) & np.uint32(0xffff0000)).astype(np.uint32).view(np.float32)
            out.append(p.astype(np.float64))
            left = left - p
        assert not left.any()                           # three parts hold all 24 bits
        return out
    x, y = (rng.integers(0, 1 << 23, 400000).astype(np.uint32) | np.uint32(0x3f800000) for _ in range(2))
    x, y = x.view(np.float32), y.view(np.float32)
    (_, x1, x2), (_, y1, y2) = parts(x), parts(y)
    small = (x1 * y2 + x2 * (y1 + y2)) / (x.astype(np.float64) * y)
    best = np.argsort(-np.abs(small))[:n]
    assert np.abs(small[best]).min() > 2.0 ** -25.7
    return x[best], y[best]


@pytest.mark.parametrize("rows,cols", [(64, 64), (128, 128), (512, 512), (192, 64), (256, 64), (64, 128), (64, 512), (2048, 512), (96, 64)])
@pytest.mark.parametrize("power_of_two", ["p", "r"])
def test_products_round_as_float32_does(pkg, rows, cols, power_of_two):
    # A matrix whose Frobenius norm rounds to 1 (one element of 1, the rest below 2^-19) is not changed by the normalisation.  Two rows and two columns of it
    # holding [[p, q], [r, 0]] have (X^T X)_01 = p q, and element (1, 1) of the next X is -r p q / 2: one product in each of the two matrix products
    # of an iteration, every other term an exact zero.  With r or p a power of two only the other product rounds.
    import torch
    short = min(rows, cols)
    n = short // 2 - 1
    x, y = hard_pairs(n, 1)
    scale, one = np.float32(2.0 ** -20), np.ones(n, np.float32)
    p, q, r = (x * scale, y * scale, one * scale) if power_of_two == "r" else (one * scale, y * scale, x * scale)
    m = np.zeros((max(rows, cols), short), np.float32)
    m[0, 0] = 1.0
    at = 2 + 2 * np.arange(n)
    m[at, at], m[at, at + 1], m[at + 1, at] = p, q, r
    if rows < cols:
        m = np.ascontiguousarray(m.T)
    ctx = pkg.Context(pkg.default_config(hidden=512, head_dim=64, n_layers=1, seq_len=32, population=2, use_muon=1))
    d = torch.from_numpy(m).cuda()
    ctx.newton_schulz(d.data_ptr(), rows, cols, 1)
    ctx.sync()
    got = d.cpu().numpy().astype(np.float64)
    got = got[at + 1, at + 1]
    want = -0.5 * r.astype(np.float64) * p * q           # exact: 48 bits
    # half a unit of the last place (2^-24) from the one rounding; the sum of the small parts is at most 2^-7 of the product and of its seven steps two reach that
    # size, each off by at most a unit of its last place (2^-31 and 2^-30); what is left out is below 2^-34: 2^-29 in all, of which the limit allows twice
    err = np.abs(got - want) / np.abs(want)
    assert err.max() <= 2.0 ** -24 * (1 + 2.0 ** -4), err.max() * 2 ** 24
    ctx.close()
