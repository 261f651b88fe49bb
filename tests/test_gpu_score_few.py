"""Few pairs are scored by two launches (score_item_kernel, score_decide_kernel): every output equals the
same pairs' in a call large enough for score_pair_kernel bit for bit -- both take the same operations per
position -- over block sizes with partial workgroups, with and without a null row, with sampling noise,
odd vocabularies, ties, rows of -inf and NaN, and inactive pairs."""

import pytest
import torch

from yapd_amd.scoring import BlockScorer

pytestmark = pytest.mark.gpu
BIG = 130  # past the limit of 128 pairs


@pytest.mark.parametrize("bl", [9, 16, 31, 32, 64])
@pytest.mark.parametrize("cfg,temperature,noise", [(0.5, 0.0, False), (0.0, 0.0, False), (1.0, 0.7, True),
                                                   (0.0, 1.3, False)])
@pytest.mark.parametrize("V", [8194, 1001])
def test_pairs_equal_those_of_a_large_call(dev, bl, cfg, temperature, noise, V):
    g = torch.Generator(device=dev).manual_seed(bl + V)
    rows = 2 * BIG if cfg > 0 else BIG
    logits = torch.full((rows, bl, (V + 7) // 8 * 8), 50.0, dtype=torch.bfloat16, device=dev)
    logits[..., :V] = torch.randn(rows, bl, V, generator=g, device=dev) * 3
    logits[1, :, 5] = logits[1, :, 900] = 30.0            # equal maxima
    logits[2, 0, :V] = float("-inf")
    logits[3, 1, :V] = float("nan")
    logits[4, 2, 7] = float("inf")
    prior = torch.rand(V, generator=g, device=dev) + 1e-3
    xt = torch.where(torch.rand(BIG, bl, generator=g, device=dev) > 0.4, V, torch.randint(
        0, V, (BIG, bl), generator=g, device=dev))
    k_step = torch.randint(0, 10, (BIG,), generator=g, device=dev)
    active = (torch.rand(BIG, generator=g, device=dev) > 0.3).to(torch.uint8)
    sc = BlockScorer(n_pairs=BIG, block_size=bl, mask_id=V, stop_id=V - 1, cfg_scale=cfg, time_shift_tau=1.0,
                     log_prior=BlockScorer.log_prior_from_prior(prior / prior.sum()), device=logits.device)
    res = []
    for n in (BIG, 128, 65, 64, 5, 1):
        r = sc(logits[: n * rows // BIG, :, :V], xt[:n], k_step[:n], layout="interleaved", active=active[:n],
               temperature=temperature, position_noise=noise, seed=11, rng_offset=3, n_pairs=n)
        res.append({k: v.clone() for k, v in vars(r).items()})
    for n, r in zip((128, 65, 64, 5, 1), res[1:]):
        for k, v in r.items():
            ref = res[0][k][:n]
            assert torch.equal(v.nan_to_num(7.5) if v.is_floating_point() else v,
                               ref.nan_to_num(7.5) if ref.is_floating_point() else ref), (n, k)


@pytest.mark.parametrize("n", [1, 5, 128])
@pytest.mark.parametrize("temperature", [0.0, 0.7])
def test_sampled_tokens_over_the_block(dev, n, temperature):
    """The sampled tokens may go to the buffer that holds the block: the decision is that of separate buffers."""
    bl, V = 16, 1001
    g = torch.Generator(device=dev).manual_seed(n)
    logits = (torch.randn(n, bl, 1008, generator=g, device=dev) * 3).to(torch.bfloat16)[..., :V]
    xt = torch.where(torch.rand(n, bl, generator=g, device=dev) > 0.4, V, 7)
    k_step = torch.full((n,), 2, dtype=torch.int64, device=dev)
    prior = torch.rand(V, generator=g, device=dev) + 1e-3
    res = []
    for over in (False, True):
        sc = BlockScorer(n_pairs=n, block_size=bl, mask_id=V, stop_id=V - 1, cfg_scale=0.0, time_shift_tau=1.0,
                         log_prior=BlockScorer.log_prior_from_prior(prior / prior.sum()), device=logits.device)
        block = xt.clone()
        if over:
            sc.out["sampled"] = block
        r = sc(logits, block, k_step, layout="interleaved", temperature=temperature, seed=11, rng_offset=3)
        res.append({k: v.clone() for k, v in vars(r).items()})
    assert res[0]["unmask"].any()
    for k, v in res[0].items():
        assert torch.equal(v, res[1][k]), k
