"""GPU parity of the sampler step: last-position logits against a float64 product, the top-k /
categorical draw bit-exactly against the CPU oracle on the SAME float32 logits and noise."""
import numpy as np
import pytest
import torch

from oracle import grpo_oracle as O

pytestmark = pytest.mark.gpu


def _draw(noise, logits, k, t):
    """Tokens, indices and values of both forms of the draw, which must agree: mj_sample_draw with its workspace
    (top_k_sampling_batched: long rows in segments) and mj_sample_top_k (one workgroup per row)."""
    import mllm_jax_amd as M
    from mllm_jax_amd import _lib
    noise = None if noise is None else noise.to(logits.device)
    tok, idx, val = M.top_k_sampling_batched(noise, logits, k=k, t=t, return_top_k=True)
    tok1, idx1, val1 = torch.empty_like(tok), torch.empty_like(idx), torch.empty_like(val)
    _lib.check(_lib.load().mj_sample_top_k(logits.data_ptr(), logits.stride(0), *logits.shape, k, t, None if noise is None else noise.data_ptr(),
                                           tok1.data_ptr(), idx1.data_ptr(), val1.data_ptr(), torch.cuda.current_stream().cuda_stream))
    assert torch.equal(tok, tok1) and torch.equal(idx, idx1) and torch.equal(val.view(torch.int32), val1.view(torch.int32))
    return tok, idx, val


def test_last_position_logits_match_float64_product():
    import mllm_jax_amd as M
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(1)
    # batch sizes either side of the 128-row tile, vocabularies that give work items of
    # 8 .. 256 columns, one full-size vocabulary
    for b, h, v, cap in [(5, 64, 1000, None), (128, 896, 5000, None), (300, 136, 2008, 30.0), (1, 8, 8, None),
                         (64, 72, 3000, None), (65, 72, 3000, None), (129, 64, 1000, 10.0), (16, 128, 152064, None),
                         (100, 64, 66000, None)]:
        hid = torch.randn(b, h, generator=g).to(torch.bfloat16)
        w = (0.2 * torch.randn(h, v, generator=g)).to(torch.bfloat16)
        out = M.last_position_logits(hid.to(dev), w.to(dev), cap)
        ref = O.lm_head_logits(hid.float().numpy(), w.float().numpy(), cap)
        assert out.dtype == torch.float32 and tuple(out.shape) == (b, v)
        np.testing.assert_allclose(out.cpu().numpy(), ref, rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("b,v,k,t", [(3, 1000, 50, 0.9), (64, 152064, 50, 1.0), (7, 129, 64, 0.7), (2, 50, 50, 1.0),
                                     (5, 4097, 1, 1.0)])
def test_top_k_draw_is_bit_exact(b, v, k, t):
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(b * 1000 + k)
    logits = (3.0 * torch.randn(b, v, generator=g)).float()
    u = torch.rand(b, k, generator=g)
    noise = -torch.log(-torch.log(u))
    tok, idx, val = _draw(noise.to(dev), logits.to(dev), k=k, t=t)
    rt, ri, rv = O.top_k_sample(logits.numpy(), k=k, t=t, noise=noise.numpy())
    np.testing.assert_array_equal(idx.cpu().numpy(), ri)
    np.testing.assert_array_equal(val.cpu().numpy(), rv)
    np.testing.assert_array_equal(tok.cpu().numpy(), rt)


@pytest.mark.parametrize("t", [3.0, 1.7, 0.6])
def test_neighbouring_floats_that_divide_to_the_same_quotient(t):
    """A cluster of adjacent float32 values around the k-th largest: after the division by t > 1
    neighbours collapse into equal quotients and the lower index must win, also for elements that
    sit a few ulps below the kernel's raw-value threshold."""
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(7)
    b, v, k = 4, 70000, 50
    x = rng.normal(-5.0, 0.5, size=(b, v)).astype(np.float32)
    for r in range(b):
        pos = rng.choice(v, size=300, replace=False)
        steps = rng.integers(0, 40, size=300)
        base = np.float32([2.0, -1.5, 1e-3, 300.0][r])
        vals = base.copy()
        cluster = np.array([np.nextafter(base, np.float32(np.inf), dtype=np.float32)] * 300, np.float32)
        for j, s_ in enumerate(steps):
            c = base
            for _ in range(int(s_)):
                c = np.nextafter(c, np.float32(np.inf), dtype=np.float32)
            cluster[j] = c
        x[r, pos] = cluster
    noise = rng.gumbel(size=(b, k)).astype(np.float32)
    tok, idx, val = _draw(torch.tensor(noise), torch.tensor(x, device=dev), k=k, t=t)
    rt, ri, rv = O.top_k_sample(x, k=k, t=t, noise=noise)
    np.testing.assert_array_equal(idx.cpu().numpy(), ri)
    np.testing.assert_array_equal(val.cpu().numpy(), rv)
    np.testing.assert_array_equal(tok.cpu().numpy(), rt)


def test_signed_zeros_and_nans_follow_the_total_order():
    """Rows of +0 / -0 / tiny values (the k-th place falls among zeros of both signs) and rows with
    NaN and infinities: selection and order are those of the IEEE total order, as in the oracle."""
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(11)
    for v, k in ((50, 34), (129, 64), (5000, 50), (70000, 50)):
        x = rng.normal(0, 1e-3, size=(6, v)).astype(np.float32)
        x[:, ::7] = 0.0
        x[:, 3::11] = -0.0
        x[3] = np.where(rng.random(v) < 0.5, 0.0, -0.0).astype(np.float32)      # nothing but zeros
        x[4, rng.integers(0, v, size=5)] = np.nan
        x[5, rng.integers(0, v, size=3)] = np.inf
        x[5, rng.integers(0, v, size=3)] = -np.inf
        tok, idx, val = _draw(None, torch.tensor(x, device=dev), k=k, t=1.3)
        rt, ri, rv = O.top_k_sample(x, k=k, t=1.3, noise=None)
        np.testing.assert_array_equal(idx.cpu().numpy(), ri)
        np.testing.assert_array_equal(val.cpu().numpy().view(np.uint32), rv.view(np.uint32))
        np.testing.assert_array_equal(tok.cpu().numpy(), rt)


def test_ties_duplicates_and_negative_values():
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(0)
    # few distinct values: the k-th largest is shared by many entries, lower indices must win
    x = rng.integers(-3, 4, size=(9, 3000)).astype(np.float32)
    x[4] = -7.0                                             # a constant row: indices 0..k-1
    x[5, 100:] = -np.inf
    noise = rng.gumbel(size=(9, 50)).astype(np.float32)
    tok, idx, val = _draw(torch.tensor(noise), torch.tensor(x, device=dev), k=50, t=1.0)
    rt, ri, rv = O.top_k_sample(x, k=50, t=1.0, noise=noise)
    np.testing.assert_array_equal(idx.cpu().numpy(), ri)
    np.testing.assert_array_equal(val.cpu().numpy(), rv)
    np.testing.assert_array_equal(tok.cpu().numpy(), rt)
    np.testing.assert_array_equal(idx[4].cpu().numpy(), np.arange(50))


def test_greedy_generator_draws_and_fused_step():
    import mllm_jax_amd as M
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(5)
    b, h, v = 32, 64, 4000
    hid = torch.randn(b, h, generator=g).to(torch.bfloat16).to(dev)
    w = (0.5 * torch.randn(h, v, generator=g)).to(torch.bfloat16).to(dev)
    logits = M.last_position_logits(hid, w)
    np.testing.assert_array_equal(M.greedy_sampling(None, logits).cpu().numpy(), logits.argmax(-1).cpu().numpy())
    gen = torch.Generator(device=dev).manual_seed(7)
    a = M.sample_next_tokens(gen, hid, w, k=50, t=1.0)
    gen.manual_seed(7)
    b2 = M.sample_next_tokens(gen, hid, w, k=50, t=1.0)
    assert torch.equal(a, b2) and a.dtype == torch.int32               # same generator state, same draw
    top = torch.topk(logits, 50, dim=-1).indices
    assert bool((top == a[:, None]).any(-1).all())                      # every draw lies inside its row's top 50
    # draws follow softmax over the top k: a sharply peaked row is (almost) always its argmax
    peaked = torch.zeros(1, v, device=dev); peaked[0, 123] = 40.0
    assert int(M.top_k_sampling_batched(gen, peaked, k=50, t=1.0)[0]) == 123
    with pytest.raises(M._lib.MjGrpoError):
        M.top_k_sampling_batched(None, logits, k=65)


def test_near_equal_logits_overflow_the_pool_and_take_the_slow_path():
    # more than 4096 logits share the 12 leading key bits of the k-th largest: the byte-wise select runs
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(2)
    x = np.full((4, 30000), 1.5, np.float32)
    x[1] += (rng.random(30000) * 1e-3).astype(np.float32)       # all inside one 12-bit bin, distinct low bits
    x[2, ::7] = 9.0                                             # 4286 equal maxima: ties beyond k
    x[3] = rng.integers(0, 3, 30000).astype(np.float32)         # three values
    noise = rng.gumbel(size=(4, 50)).astype(np.float32)
    tok, idx, val = _draw(torch.tensor(noise), torch.tensor(x, device=dev), k=50, t=1.0)
    rt, ri, rv = O.top_k_sample(x, k=50, t=1.0, noise=noise)
    np.testing.assert_array_equal(idx.cpu().numpy(), ri)
    np.testing.assert_array_equal(val.cpu().numpy(), rv)
    np.testing.assert_array_equal(tok.cpu().numpy(), rt)


@pytest.mark.parametrize("v,ld", [(4096, 4096), (16381, 16384), (16384, 16387), (16385, 16392), (32769, 32769), (49153, 49160)])
def test_rows_cut_into_segments_draw_like_whole_rows(v, ld):
    """Vocabularies either side of a segment's 16384 elements, rows that are not 16-byte aligned, the
    largest values at the segments' ends, NaNs, ties across segments and a row whose ties overflow a
    segment's pool: bit for bit the oracle's choice."""
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(v)
    k = 64
    x = rng.normal(0, 1, size=(6, ld)).astype(np.float32)
    x[1, [0, v - 1, v // 2, min(16383, v - 1)]] = 9.0
    x[2, v - 3:v] = np.float32(7.0)
    x[2, v:] = 99.0                                                  # padding of the row: never looked at
    x[3, rng.integers(0, v, 70)] = np.nan
    x[4, ::97] = 5.0                                                 # more than k equal maxima, spread over the segments
    x[5] = 1.0
    noise = rng.gumbel(size=(6, k)).astype(np.float32)
    lg = torch.tensor(x, device=dev)[:, :v]
    tok, idx, val = _draw(torch.tensor(noise), lg, k=k, t=0.9)
    rt, ri, rv = O.top_k_sample(x[:, :v], k=k, t=0.9, noise=noise)
    np.testing.assert_array_equal(idx.cpu().numpy(), ri)
    np.testing.assert_array_equal(val.cpu().numpy().view(np.uint32), rv.view(np.uint32))
    rows = [0, 1, 2, 4, 5]                                           # what argmax makes of NaN scores is not at issue here
    np.testing.assert_array_equal(tok.cpu().numpy()[rows], rt[rows])


@pytest.mark.parametrize("b,h,v,cap", [(1, 8, 8, None), (1, 24, 264, 30.0), (2, 56, 1000, None), (2, 72, 256, 10.0), (1, 136, 2008, None),
                                       (2, 904, 5000, None),
                                       # pieces of 64 columns in eight wavefronts, of 64 and 128, whole ones of 256, and even
                                       # shares of one, two and three rounds; pitches (v + 16) with and without shared lines
                                       (1, 40, 16368, None), (2, 40, 16376, None), (1, 24, 36848, None), (1, 24, 36880, None), (2, 24, 45040, None),
                                       (2, 24, 45064, None), (1, 24, 65520, None), (2, 24, 65536, None), (1, 24, 65544, 30.0), (2, 24, 72008, None),
                                       (1, 24, 131056, None), (2, 136, 131080, None)])
def test_one_or_two_rows_on_the_vector_alus(b, h, v, cap):
    """k_logits_few: odd counts of 8-row groups, columns either side of a workgroup's 256 and of each split, softcap;
    a row pitch of W and of hidden past their lengths.  The bound is float32 summation: h products of at most
    0.2 * 4 * 4 in magnitude, one rounding of 2^-24 of the partial sum each."""
    import mllm_jax_amd as M
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(h + v)
    hid = torch.randn(b, h + 8, generator=g).to(torch.bfloat16)
    w = (0.2 * torch.randn(h, v + 16, generator=g)).to(torch.bfloat16)
    w[:, v:] = float("nan")                                          # padding: never looked at
    hid[:, h:] = float("nan")
    out = M.last_position_logits(hid.to(dev)[:, :h], w.to(dev)[:, :v], cap)
    ref = O.lm_head_logits(hid[:, :h].float().numpy(), w[:, :v].float().numpy(), cap)
    np.testing.assert_allclose(out.cpu().numpy(), ref, rtol=1e-5, atol=h * 3.2 * 2.0 ** -24 * 4)


def test_a_row_whose_last_segment_would_be_a_single_logit():
    """4095 * 16384 + 1 logits, all negative, the largest at the very end: cut into 4096 segments the last one
    would hold one logit.  Distinct values, so the top k of the row is that of torch.topk."""
    v = 4095 * 16384 + 1
    row = torch.full((1, v), -5.0, device="cuda:0")
    at = torch.arange(63, device="cuda:0") * 1000003 + 17
    row[0, at] = -1.0 - 0.01 * torch.arange(63, device="cuda:0")
    row[0, v - 1] = -0.5
    tok, idx, val = _draw(None, row, k=64, t=1.0)
    assert int(tok[0]) == v - 1
    assert idx[0].tolist() == [v - 1] + at.tolist()
    assert torch.equal(val[0], row[0, idx[0].long()])


@pytest.mark.parametrize("b", [1, 2, 3])
@pytest.mark.parametrize("h", [8, 24, 40, 136, 144])
def test_infinities_in_hidden_stay_infinities(b, h):
    """An infinity in the last eight hidden values gives +-inf logits and no NaN (no entry of W is zero), for
    lengths that end in the middle of a group of sixteen k-rows and for those that do not; three rows take
    the matrix form."""
    import mllm_jax_amd as M
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(h)
    hid = torch.randn(b, h, generator=g).to(torch.bfloat16)
    w = torch.randn(h, 520, generator=g).to(torch.bfloat16)
    w[w == 0] = 1.0
    hid[0, h - 3] = float("inf")
    out = M.last_position_logits(hid.to(dev), w.to(dev)).cpu()
    expect = torch.where(w[h - 3] > 0, float("inf"), float("-inf"))
    assert torch.equal(out[0], expect)
    assert bool(torch.isfinite(out[1:]).all())


@pytest.mark.filterwarnings("ignore:overflow encountered in divide")
@pytest.mark.parametrize("v,k", [(8200, 64), (16388, 50), (40001, 64), (152064, 64), (152064, 1), (70 * 16384 + 5, 3), (1 << 21, 64)])
def test_masked_blocks_and_crowded_segments(v, k):
    """Segments in which more elements reach the threshold than the pool holds: blocks of -inf and of the
    type's lowest value that fill whole segments, rows with a handful of unmasked logits, one value everywhere,
    ties in the middle of a segment, two neighbouring floats, NaNs; also more segments than k and than a
    wavefront has lanes, and lists whose words overflow the draw's pool.  Bit for bit the oracle's choice."""
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(v + k)
    x = rng.normal(0, 2, size=(11, v)).astype(np.float32)
    low = np.finfo(np.float32).min
    x[1, v // 4:v // 4 + 40000] = -np.inf
    x[2, v // 4:v // 4 + 40000] = low
    x[3] = -np.inf
    x[3, rng.choice(v, size=40, replace=False)] = rng.normal(0, 2, size=40).astype(np.float32)
    x[4] = low
    x[4, v - 30:] = rng.normal(0, 2, size=30).astype(np.float32)
    x[5] = -1.25
    x[6, ::3] = 3.0                                                     # a third of the row, larger than most others
    x[7] = np.where(rng.random(v) < 0.5, np.float32(2.0), np.nextafter(np.float32(2.0), np.float32(3.0)))
    x[8, 700:] = low                                                    # the edge of a masked block
    x[9, 1000:] = -np.inf
    x[9, ::5] = np.round(x[9, ::5])                                     # few distinct values above it
    x[10, :20000] = np.nan
    noise = rng.gumbel(size=(11, k)).astype(np.float32)
    tok, idx, val = _draw(torch.tensor(noise), torch.tensor(x, device=dev), k=k, t=0.9)
    rt, ri, rv = O.top_k_sample(x, k=k, t=0.9, noise=noise)
    np.testing.assert_array_equal(idx.cpu().numpy(), ri)
    np.testing.assert_array_equal(val.cpu().numpy().view(np.uint32), rv.view(np.uint32))
    np.testing.assert_array_equal(tok.cpu().numpy()[:10], rt[:10])       # what argmax makes of NaN scores is not at issue here


@pytest.mark.filterwarnings("ignore:overflow encountered in divide")
@pytest.mark.parametrize("v", [3000, 40000])
@pytest.mark.parametrize("t,scale", [(2e-38, 1.0), (2e-38, 30.0), (3e38, 1e-3), (3e38, 1e-6), (1e20, 1e-25)])
def test_quotients_that_overflow_or_lose_their_digits(v, t, scale):
    """logits / t past the largest float (many equal +inf, lower index first) or among the denormals (logits far
    apart share a quotient, or become zeros): the order is that of the quotients, not of the logits."""
    rng = np.random.default_rng(v)
    x = (scale * rng.normal(0, 2, size=(3, v))).astype(np.float32)
    x[2] = -np.abs(x[2])
    noise = rng.gumbel(size=(3, 50)).astype(np.float32)
    tok, idx, val = _draw(torch.tensor(noise), torch.tensor(x, device="cuda:0"), k=50, t=t)
    rt, ri, rv = O.top_k_sample(x, k=50, t=t, noise=noise)
    np.testing.assert_array_equal(idx.cpu().numpy(), ri)
    np.testing.assert_array_equal(val.cpu().numpy().view(np.uint32), rv.view(np.uint32))
    np.testing.assert_array_equal(tok.cpu().numpy(), rt)
