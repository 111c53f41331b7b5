"""The Newton-Schulz products on bf16 parts of float32 operands, against the iteration in 64 bits: one to many chunks of k, odd numbers of
them, both tile sizes, both operand orders, and the shapes next to the kernel's (sides that are not multiples of 64)."""
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
    # float32 products err by up to 9.1e-7 at these sizes, bf16 parts by 6.0e-7; a partial product left out (2^-18 and more) by 4e-6
    assert err < 1.5e-6, err
    ctx.close()
