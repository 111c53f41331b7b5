"""The rank-one term of the MLP's up projection as one more k-step (egg_rank1_kstep), against the oracle: losses of sampled members with saturated norms and
the smallest sigma that takes the form, where a few tokens in a hundred have sums that need the third digit; and masks and sigmas just outside it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,head_dim,seq,population,sigma,mask", [
    (64, 32, 32, 66, 4, 15), (64, 32, 128, 514, 4, 15), (64, 32, 32, 66, 3, 15), (128, 32, 64, 34, 5, 15), (128, 64, 64, 514, 5, 15),
    (256, 64, 64, 770, 6, 15), (256, 64, 64, 34, 6, 15), (256, 64, 128, 258, 6, 15), (512, 64, 64, 10, 7, 15), (512, 64, 64, 514, 7, 15),
    (128, 32, 64, 514, 6, 31), (64, 32, 32, 66, 4, 7)],
    ids=lambda v: str(v))
def test_up_projection_noise(pkg, orc, hidden, head_dim, seq, population, sigma, mask):
    import torch
    kw = dict(hidden=hidden, head_dim=head_dim, seq_len=seq, population=population, n_layers=1, fixed_point=3, sigma_shift=sigma - 3, sigma_shift_vector=7, noise_mask=mask)
    members = sorted({0, 1, 2, 3, population // 3, population // 2, population - 2, population - 1})
    ocfg, rng = orc.config(**kw), np.random.default_rng(hidden + sigma)
    data, model = orc.zipf_bytes(1 << 16), orc.init_model(orc.config(**kw), 42)
    for t in orc.tensor_table(ocfg):
        if not t["is_matrix"]:
            gain = t["name"].startswith("ln_") and "bias" not in t["name"]
            model[t["offset"]:t["offset"] + t["cols"]] = rng.integers(100, 127, t["cols"]) * rng.choice([-1, 1], t["cols"]) if gain else rng.integers(-20, 21, t["cols"])
    ctx = pkg.Context(pkg.default_config(**kw))
    ctx.model_upload(model)
    d_data, loss = torch.from_numpy(data).cuda(), torch.zeros(population, dtype=torch.int32, device="cuda")
    ctx.population_forward(d_data.data_ptr(), len(data), 7, 99, 0, population, loss.data_ptr())
    ctx.sync()
    got = loss.cpu().numpy()
    ref = [orc.forward_member(ocfg, model, data, 7, 99, m) for m in members]
    assert [int(got[m]) for m in members] == [r[0] if isinstance(r, tuple) else r for r in ref]
    ctx.close()
