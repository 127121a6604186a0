"""The pass that adds up the logits' statistics, at chunk sizes either side of its block's change from 16 to 32 tokens, and
the pass over the stored logits behind the running maximum in shares of a row: against torch in float32."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("temperature", [1.0, 0.7])
@pytest.mark.parametrize("n", [1, 15, 17, 4095, 4096, 4129])
def test_sums_over_vocabulary_tiles(n, temperature):
    """320 parts of which the last two are partly filled; masked tokens in runs that end inside a block of 16 and 32."""
    import mllm_jax_amd as M
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(n)
    h, v = 32, 40840
    hid = torch.randn(n, h, generator=g, device=dev).to(torch.bfloat16)
    w = (torch.randn(h, v, generator=g, device=dev) / h ** 0.5).to(torch.bfloat16)
    y = torch.randint(0, v, (n,), generator=g, device=dev)
    mask = ((torch.arange(n, device=dev) // 21) % 2 == 0).float()
    tv = float(mask.sum())
    met, (dh, _) = M.grpo_loss_value_and_grad(hid, w, y, None, torch.ones(n, device=dev), mask, total_valid_token_count=tv,
                                              temperature=temperature, return_token_entropy=True)
    z = hid.float() @ w.float()
    lp = torch.log_softmax(z, -1)
    p = torch.softmax(z / temperature, -1)
    ent = -(p * torch.log_softmax(z / temperature, -1)).sum(-1)
    # float32 sums of 40840 terms on either side: 1e-5 of values near 11
    assert (met["per_token_logps"] - lp.gather(1, y[:, None])[:, 0] / temperature).abs().max().item() <= 2e-4
    assert (met["token_entropy"] - ent).abs().max().item() <= 2e-4
    # d_hidden = -(1 / T tv) (W_y - p W^T), bf16 operands: 2^-8 of its norm, twice that allowed
    ref = -(w.float().index_select(1, y).t() - torch.softmax(z, -1) @ w.float().t()) * (mask / (temperature * tv))[:, None]
    assert ((dh.float() - ref).norm() / ref.norm()).item() <= 2.0 ** -7
    assert not dh[mask == 0].any()


@pytest.mark.parametrize("n,v", [(3, 8), (40, 2048), (2048, 2056), (2100, 16400), (4097, 4104)])
def test_stored_logits_in_shares_of_a_row(n, v):
    """An entropy bonus: every row goes through k_dz, in eight, four or one share; vocabularies below a share, at its end
    and past it."""
    import mllm_jax_amd as M
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(v)
    h, coef = 24, 0.3
    hid = torch.randn(n, h, generator=g, device=dev).to(torch.bfloat16)
    w = (torch.randn(h, v, generator=g, device=dev) / h ** 0.5).to(torch.bfloat16)
    y = torch.randint(0, v, (n,), generator=g, device=dev)
    ones = torch.ones(n, device=dev)
    _, (dh, dw) = M.grpo_loss_value_and_grad(hid, w, y, None, ones, ones, total_valid_token_count=float(n), entropy_coef=coef)
    a, b = hid.float().requires_grad_(), w.float().requires_grad_()
    lp = torch.log_softmax(a @ b, -1)
    loss = -(torch.exp(lp.gather(1, y[:, None])[:, 0] - lp.gather(1, y[:, None])[:, 0].detach())).mean() + coef * (lp.exp() * lp).sum(-1).mean()
    ga, gb = torch.autograd.grad(loss, [a, b])
    # dZ is rounded to bf16 from half-precision logits (2^-11 each) and meets bf16 operands (2^-9): 2^-7 bounds the norm
    assert ((dh.float() - ga).norm() / ga.norm()).item() <= 2.0 ** -7
    assert ((dw - gb).norm() / gb.norm()).item() <= 2.0 ** -7
