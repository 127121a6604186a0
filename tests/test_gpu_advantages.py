"""GPU: the advantage estimators against the reference tests' known answers
(tests/test_advantage_estimators.py:19-106, restated) and against the CPU oracle on random batches."""
import numpy as np
import pytest
import torch

from oracle import grpo_oracle as O

pytestmark = pytest.mark.gpu
R5 = np.asarray([1.0, 2.0, 3.0, 10.0, 20.0], np.float32)
G5 = np.asarray([0, 0, 0, 1, 1], np.int32)


def _d(x):
    return torch.as_tensor(np.asarray(x)).to("cuda:0")


def test_reference_known_answers_on_device():
    import mllm_jax_amd as M
    r4 = np.asarray([0.0, 1.0, 2.0, 3.0], np.float32)
    out = M.compute_global_normalized_advantages(rewards=_d(r4), eps=1e-4)
    np.testing.assert_allclose(out.cpu().numpy(), ((r4 - r4.mean()) / (r4.std() + 1e-4)).astype(np.float32), rtol=0, atol=1e-6)
    out = M.compute_global_normalized_advantages(rewards=_d([-100.0, 0.0, 100.0]), eps=1e-6, clip_range=0.5).cpu().numpy()
    assert (out <= 0.5).all() and (out >= -0.5).all()
    out = M.compute_rloo_advantages_by_group_id(rewards=_d(R5), group_ids=_d(G5), whiten=False, eps=1e-6)
    np.testing.assert_allclose(out.cpu().numpy(), [-1.5, 0.0, 1.5, -10.0, 10.0], rtol=0, atol=1e-6)
    out = M.compute_rloo_advantages_by_group_id(rewards=_d(R5), group_ids=_d(G5), whiten=True, eps=1e-6).cpu().numpy()
    assert abs(float(out.mean())) < 1e-5 and float(out.std()) > 0.5
    grpo = M.compute_grpo_advantages_by_group_id(rewards=_d(R5), group_ids=_d(G5), eps=1e-4)
    glob = M.compute_global_normalized_advantages(rewards=_d(R5), eps=1e-4)
    out = M.compute_dapo_advantages_by_group_id(rewards=_d(R5), group_ids=_d(G5), eps=1e-4, alpha=0.5)
    np.testing.assert_allclose(out.cpu().numpy(), (grpo + 0.5 * glob).cpu().numpy(), rtol=0, atol=1e-6)
    out = M.compute_reinforce_plus_plus_advantages_by_group_id(rewards=_d(R5), group_ids=_d(G5), eps=1e-4)
    exp = M.compute_rloo_advantages_by_group_id(rewards=_d(R5), group_ids=_d(G5), eps=1e-4, whiten=True)
    np.testing.assert_allclose(out.cpu().numpy(), exp.cpu().numpy(), rtol=0, atol=1e-6)
    out = M.build_token_rewards_from_final(rewards=_d([1.0, 2.0]), completion_mask=_d([[1, 1, 0], [0, 1, 1]]))
    np.testing.assert_allclose(out.cpu().numpy(), [[0.0, 1.0, 0.0], [0.0, 0.0, 2.0]], rtol=0, atol=1e-6)
    adv, ret = M.compute_gae_advantages(rewards=_d([1.0]), values=_d(np.zeros((1, 3), np.float32)),
                                        completion_mask=_d(np.ones((1, 3), np.float32)), gamma=1.0, gae_lambda=1.0,
                                        normalize=False, eps=1e-6)
    np.testing.assert_allclose(adv.cpu().numpy(), np.ones((1, 3)), rtol=0, atol=1e-6)
    np.testing.assert_allclose(ret.cpu().numpy(), np.ones((1, 3)), rtol=0, atol=1e-6)
    adv, _ = M.compute_gae_advantages(rewards=_d([1.0]), values=_d(np.zeros((1, 3), np.float32)),
                                      completion_mask=_d([[0.0, 1.0, 1.0]]), gamma=1.0, gae_lambda=1.0,
                                      normalize=False, eps=1e-6)
    np.testing.assert_allclose(adv.cpu().numpy(), [[0.0, 1.0, 1.0]], rtol=0, atol=1e-6)


@pytest.mark.parametrize("b", [1, 7, 128, 3000])
def test_random_batches_match_oracle(b):
    import mllm_jax_amd as M
    rng = np.random.default_rng(b)
    r = rng.standard_normal(b).astype(np.float32) * 3 + 1
    gid = rng.integers(-4, max(b // 5, 1), b).astype(np.int32)
    kw = dict(rtol=2e-6, atol=2e-6)
    np.testing.assert_allclose(M.compute_global_normalized_advantages(rewards=_d(r), eps=1e-3).cpu().numpy(),
                               O.global_normalized_advantages(r, 1e-3), **kw)
    for whiten in (False, True):
        np.testing.assert_allclose(
            M.compute_rloo_advantages_by_group_id(rewards=_d(r), group_ids=_d(gid), whiten=whiten, clip_range=1.5).cpu().numpy(),
            O.rloo_advantages(r, gid, whiten=whiten, clip_range=1.5), **kw)
    np.testing.assert_allclose(M.compute_dapo_advantages_by_group_id(rewards=_d(r), group_ids=_d(gid), alpha=0.3).cpu().numpy(),
                               O.dapo_advantages(r, gid, alpha=0.3), rtol=1e-5, atol=1e-5)
    np.testing.assert_allclose(M.compute_grpo_advantages_by_group_id(rewards=_d(r), group_ids=_d(gid)).cpu().numpy(),
                               O.grpo_advantages(r, gid), rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("b,t,normalize,clip", [(1, 1, False, None), (5, 17, True, None), (64, 130, True, 2.0), (300, 33, False, 0.5)])
def test_gae_matches_oracle(b, t, normalize, clip):
    import mllm_jax_amd as M
    rng = np.random.default_rng(b * 100 + t)
    r = rng.standard_normal(b).astype(np.float32)
    v = rng.standard_normal((b, t)).astype(np.float32) * 0.5
    start = rng.integers(0, t, b); length = rng.integers(0, t + 1, b)
    ar = np.arange(t)[None]
    m = ((ar >= start[:, None]) & (ar < (start + length)[:, None])).astype(np.float32)    # some rows empty
    adv, ret = M.compute_gae_advantages(rewards=_d(r), values=_d(v), completion_mask=_d(m), gamma=0.97, gae_lambda=0.9,
                                        normalize=normalize, eps=1e-4, clip_range=clip)
    ra, rr = O.gae_advantages(r, v, m, 0.97, 0.9, normalize, 1e-4, clip)
    np.testing.assert_allclose(ret.cpu().numpy(), rr, rtol=1e-5, atol=1e-5)
    np.testing.assert_allclose(adv.cpu().numpy(), ra, rtol=2e-5, atol=2e-5)


def test_argument_errors_mirror_the_reference():
    import mllm_jax_amd as M
    with pytest.raises(ValueError):
        M.compute_global_normalized_advantages(rewards=_d(R5), eps=0.0)
    with pytest.raises(ValueError):
        M.compute_rloo_advantages_by_group_id(rewards=_d(R5), group_ids=_d(G5[:4]))
    with pytest.raises(ValueError):
        M.compute_dapo_advantages_by_group_id(rewards=_d(R5), group_ids=_d(G5), alpha=-1.0)
    with pytest.raises(ValueError):
        M.compute_global_normalized_advantages(rewards=_d(R5), clip_range=0.0)
    with pytest.raises(ValueError):
        M.compute_gae_advantages(rewards=_d(R5), values=_d(np.zeros((5, 3), np.float32)), completion_mask=_d(np.zeros((5, 4), np.float32)))
    with pytest.raises(RuntimeError):
        M.compute_global_normalized_advantages(rewards=torch.tensor(R5))


@pytest.mark.parametrize("t", [3, 4, 255, 256, 257, 513, 1024])
@pytest.mark.parametrize("gamma,lam", [(1.0, 0.95), (1.0, 1.0), (0.9, 0.0)])
def test_gae_blocks_of_256_tokens(t, gamma, lam):
    """Sequence lengths either side of a lane's four tokens and of a 256-token block; completions that end
    in the last block, in an earlier one, in the middle of a lane's tokens, or nowhere."""
    import mllm_jax_amd as M
    rng = np.random.default_rng(t)
    b = 7
    r = rng.standard_normal(b).astype(np.float32)
    v = rng.standard_normal((b, t)).astype(np.float32)
    end = np.array([t, t - 1, max(t // 2, 1), 1, 0, max(t - 255, 1), max(t - 257, 1)])
    m = ((np.arange(t)[None] >= end[:, None] // 3) & (np.arange(t)[None] < end[:, None])).astype(np.float32)
    adv, ret = M.compute_gae_advantages(rewards=_d(r), values=_d(v), completion_mask=_d(m), gamma=gamma, gae_lambda=lam,
                                        normalize=False)
    ra, rr = O.gae_advantages(r, v, m, gamma, lam, False, 1e-4, None)
    # both walk up to t float32 steps; each adds a rounding of 2^-24 of a running value of a few sigma
    tol = dict(rtol=1e-5, atol=max(1e-5, t * 2.0 ** -24 * 8))
    np.testing.assert_allclose(ret.cpu().numpy(), rr, **tol)
    np.testing.assert_allclose(adv.cpu().numpy(), ra, **tol)


@pytest.mark.parametrize("b", [15, 16, 17, 255, 257, 1039])
def test_batches_across_workgroups(b):
    """Batch sizes either side of a workgroup's samples; one group, singletons, and ragged groups."""
    import mllm_jax_amd as M
    rng = np.random.default_rng(b)
    r = rng.standard_normal(b).astype(np.float32)
    for gid in (np.zeros(b, np.int32), np.arange(b, dtype=np.int32), rng.integers(0, max(b // 7, 1), b).astype(np.int32)):
        kw = dict(rtol=1e-5, atol=1e-5)
        np.testing.assert_allclose(M.compute_grpo_advantages_by_group_id(rewards=_d(r), group_ids=_d(gid)).cpu().numpy(),
                                   O.grpo_advantages(r, gid), **kw)
        np.testing.assert_allclose(M.compute_rloo_advantages_by_group_id(rewards=_d(r), group_ids=_d(gid), whiten=b > 16, clip_range=1.0).cpu().numpy(),
                                   O.rloo_advantages(r, gid, whiten=b > 16, clip_range=1.0), **kw)
        np.testing.assert_allclose(M.compute_dapo_advantages_by_group_id(rewards=_d(r), group_ids=_d(gid), clip_range=0.9).cpu().numpy(),
                                   O.dapo_advantages(r, gid, clip_range=0.9), **kw)


@pytest.mark.parametrize("b", [1, 200, 256, 257, 1024, 5000, 65536])
def test_global_advantages_in_place(b):
    """advantages == rewards, up to the largest batch: what the call gives for separate buffers."""
    from mllm_jax_amd import _lib
    rng = np.random.default_rng(b)
    r = (3.0 + rng.standard_normal(b)).astype(np.float32)
    x = _d(r)
    _lib.check(_lib.load().mj_grpo_advantages(1, x.data_ptr(), None, x.data_ptr(), b, 1e-4, 0.0, 0, 1.5,
                                              torch.cuda.current_stream().cuda_stream))
    np.testing.assert_allclose(x.cpu().numpy(), O.global_normalized_advantages(r, eps=1e-4, clip_range=1.5), rtol=1e-5, atol=1e-5)


def test_vectors_that_are_read_in_place_give_what_converted_ones_give():
    """Contiguous float32 rewards and int32 ids go to the kernel as they are; anything else is converted first."""
    import mllm_jax_amd as M
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(3)
    r = torch.randn(37, generator=g).to(dev)
    ids = (torch.arange(37, dtype=torch.int32) // 5).to(dev)
    wide = torch.stack([r, r + 1], 1)
    for fn in (M.compute_grpo_advantages_by_group_id, M.compute_rloo_advantages_by_group_id, M.compute_dapo_advantages_by_group_id):
        plain = fn(rewards=r, group_ids=ids)
        assert plain.data_ptr() != r.data_ptr()
        for rr, gg in ((r.double(), ids), (wide[:, 0], ids.long()), (r, ids.cpu()), (torch.nn.Parameter(r), ids)):
            assert torch.equal(plain, fn(rewards=rr, group_ids=gg))
        with pytest.raises(ValueError):
            fn(rewards=r, group_ids=ids[:36])
        with torch.cuda.stream(torch.cuda.Stream()):
            other = fn(rewards=r, group_ids=ids)
        torch.cuda.synchronize()
        assert torch.equal(plain, other)
