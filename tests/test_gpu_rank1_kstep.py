"""The rank-one term as one more k-step of the W-stationary linear layer, against integer sums: every noise value, sums whose high part needs the
second digit (rows that follow the noise's signs), the largest and smallest of them, odd member counts, and masks on both sides of the form."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _noise(orc, seed, n, mask):
    return orc.noise_vec(seed & 0xFFFFFFFF, n, mask, 0).astype(np.int64)


@pytest.mark.parametrize("members,T,K", [(3, 32, 512), (257, 32, 512), (5, 96, 512), (3, 64, 256), (513, 32, 256)])
@pytest.mark.parametrize("mask,sigma", [(15, 7), (7, 6), (15, 6), (15, 9), (31, 7), (0, 7)])
def test_perturbed_linear(pkg, orc, members, T, K, mask, sigma):
    import torch
    N, seed, off_a, off_b = 512, 77, 200, 201
    ctx = pkg.Context(pkg.default_config(population=2, seq_len=32, noise_mask=mask, fixed_point=4, sigma_shift=sigma - 4))
    rng = np.random.default_rng(members + K + mask)
    x = rng.integers(-127, 128, (members, T, K)).astype(np.int8)
    W = rng.integers(-127, 128, (K, N)).astype(np.int8)
    for m in range(0, members, 2):                     # rows that follow (or oppose) their noise in all, most or half of the columns
        B = _noise(orc, seed + m // 2 + off_b, K, mask)
        for t, (sign, share) in enumerate([(1, 1.0), (-1, 1.0), (1, 0.75), (-1, 0.6), (1, 0.52)]):
            follow = rng.random(K) < share
            x[m, 3 * t + 1] = np.where(follow, sign * 127 * np.sign(B), x[m, 3 * t + 1])
    blocked = W.reshape(K // 4, 4, N).transpose(0, 2, 1).copy()
    d_x, d_w = torch.from_numpy(x).cuda(), torch.from_numpy(blocked).cuda()
    for own in (False, True):
        for shift, out in ((8, np.int8), (9, np.int8), (8, np.int32)):
            y = torch.empty((members, T, N), dtype=torch.int8 if out == np.int8 else torch.int32, device="cuda")
            call = ctx.perturbed_linear_own_noise if own else ctx.perturbed_linear
            ptr = (None, y.data_ptr()) if out == np.int8 else (y.data_ptr(), None)
            call(d_x.data_ptr(), d_w.data_ptr(), members, T, K, N, seed, off_a, off_b, shift, *ptr)
            ctx.sync()
            got = y.cpu().numpy()
            for m in sorted({0, 1, 2, members // 2, members - 1}):
                ps, ns = (seed + m, 1) if own else (seed + m // 2, -1 if m & 1 else 1)
                xm = x[m].astype(np.int64)
                sb = xm @ _noise(orc, ps + off_b, K, mask)
                acc = xm @ W.astype(np.int64) + ((sb[:, None] * (_noise(orc, ps + off_a, N, mask) * ns)[None, :]) >> sigma)
                ref = acc >> shift
                if out == np.int8:
                    ref = np.clip(ref, -127, 127)
                assert np.array_equal(got[m], ref.astype(out)), (own, shift, out, m)
    ctx.close()
