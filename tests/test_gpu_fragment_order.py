"""Operands that the product kernels read in fragment order (blocks of 16 rows x 32 k): sizes either side of a block, a
slice of 64 and a tile, few and odd numbers of slices, and live tokens that end inside any of them, against the CPU oracle."""
import numpy as np
import pytest
import torch

from oracle import grpo_oracle as O

pytestmark = pytest.mark.gpu

# Each gradient is a sum of products of two operands rounded to bf16 (relative error at most 2^-9 each), so its norm
# is off by at most 2^-8; a factor of two on top for the float32 sums and the one-hot entries.
RTOL = 2.0 ** -7


def _rel(a, b, axis=None):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return np.linalg.norm(a - b, axis=axis) / np.maximum(np.linalg.norm(b, axis=axis), 1e-30)


@pytest.mark.parametrize("skip", [False, True])
@pytest.mark.parametrize("n,h,v", [(1, 8, 8), (16, 24, 264), (17, 16, 40), (63, 40, 72), (64, 264, 64), (65, 136, 520),
                                   (129, 72, 1000), (193, 248, 296), (256, 256, 256), (257, 280, 776), (321, 8, 2056),
                                   (600, 520, 1064)])
def test_edges_of_blocks_slices_and_tiles(n, h, v, skip):
    import mllm_jax_amd as M
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(n * 7 + h)
    hid = torch.randn(n, h, generator=g).to(torch.bfloat16)
    w = (torch.randn(h, v, generator=g) / np.sqrt(h)).to(torch.bfloat16)
    y = torch.randint(0, v, (n,), generator=g)
    adv = 1.0 + torch.rand(n, generator=g)
    mask = (torch.rand(n, generator=g) < 0.7).float()
    mask[0] = mask[n - 1] = 1.0
    tv = float(mask.sum())
    met, (dh, dw) = M.grpo_loss_value_and_grad(hid.to(dev), w.to(dev), y.to(dev), None, adv.to(dev), mask.to(dev),
                                               total_valid_token_count=tv, skip_masked=skip)
    ref = O.grpo_loss(hid.float().numpy(), w.float().numpy(), y.numpy(), None, adv.numpy(), mask.numpy(),
                      total_valid_token_count=tv)
    np.testing.assert_allclose(met["per_token_logps"].cpu().numpy(), ref["per_token_logps"], atol=1e-3, rtol=0)
    dh, dw = dh.float().cpu().numpy(), dw.cpu().numpy()
    assert _rel(dh, ref["d_hidden"]) <= RTOL and _rel(dw, ref["d_lm_head"]) <= RTOL
    # no token and no hidden column of its own is wrong, at the edges in particular
    assert (_rel(dh, ref["d_hidden"], 1)[mask.numpy() != 0] <= 4 * RTOL).all() and not dh[mask.numpy() == 0].any()
    assert (_rel(dw, ref["d_lm_head"], 1) <= 4 * RTOL).all()


@pytest.mark.parametrize("n,h,v,cap", [(1100, 1032, 152064, 0.0), (2049, 1000, 80008, 0.0), (300, 4088, 131080, 20.0), (401, 8160, 50000, 0.0)])
def test_logits_of_hidden_in_fragment_order_are_the_same_bits(n, h, v, cap):
    """Ragged tokens, hidden sizes that end inside a block of 32 and a slice of 64 with an odd and an even number of
    slices: a workspace without room for the reordered copy takes the path that reads hidden in place."""
    import ctypes as C

    from mllm_jax_amd import _lib
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(h)
    hid = torch.randn(n, h + 8, generator=g, device=dev).to(torch.bfloat16)       # row pitch of its own
    hid[:, h:] = float("nan")
    w = (torch.randn(h, v, generator=g, device=dev) / np.sqrt(h)).to(torch.bfloat16)
    y = torch.randint(0, v, (n,), generator=g, device=dev, dtype=torch.int32)
    ones = torch.ones(n, device=dev)
    d = _lib.MjGrpoDesc()
    d.n_tokens, d.hidden, d.vocab, d.ld_hidden, d.ld_w = n, h, v, h + 8, v
    d.eps_low = d.eps_high = 0.2
    d.temperature, d.softcap, d.inv_total_valid_tokens, d.grad_loss_scale = 1.0, cap, 1.0 / n, 1.0
    full, _ = _lib.workspace_bytes(d)
    copy = -(-n // 256) * 256 * (-(-h // 64) * 64) * 2
    runs = []
    for nbytes in (full, full - copy):
        ws = torch.full((nbytes,), 255, dtype=torch.uint8, device=dev)             # NaNs wherever it is read unwritten
        logp, lse, ent, loss = (torch.empty(k, device=dev) for k in (n, n, n, 2))
        _lib.check(_lib.load().mj_grpo_forward(C.byref(d), hid.data_ptr(), w.data_ptr(), y.data_ptr(), None, ones.data_ptr(), ones.data_ptr(),
                                               logp.data_ptr(), lse.data_ptr(), ent.data_ptr(), loss.data_ptr(), ws.data_ptr(), nbytes,
                                               torch.cuda.current_stream().cuda_stream))
        runs.append((logp, lse, ent, loss))
    assert all(torch.equal(a, b) for a, b in zip(*runs))
    z = hid[:, :h].float() @ w.float()
    z = cap * torch.tanh(z / cap) if cap else z
    ref = torch.log_softmax(z, -1).gather(1, y.long()[:, None])[:, 0]
    assert (runs[0][0] - ref).abs().max().item() <= 1e-3
