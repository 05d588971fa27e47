"""The prefill attention kernels (hip/prefill.hip pf_attn, pf_attn16) on the
GPU, each forced, against plain PyTorch in 64 bits: query counts and start
positions around the edges of their tiles, cache rows past the last position
that hold infinities and NaN, queries of extreme magnitude, and a key row with
an infinity."""
import pytest

pytestmark = pytest.mark.gpu

H, TMAX, L, B = 3, 330, 2, 2
D = 64 * H


@pytest.fixture(scope='module')
def engine():
    import torch
    if not torch.cuda.is_available():
        pytest.skip('no GPU')
    from vesta.gpt2 import VestaGPT2
    from vesta.weights import GPT2Shape, RandomGPT2
    return VestaGPT2(RandomGPT2(GPT2Shape(L, D, H, 4 * D, vocab=203), 5), batch=1, tmax=32, engine='layered')._pf


def _run(e, kernel, Q, k, v, t0, P):
    import torch
    from vesta import prefill as pf
    M, MT = Q.shape[0], pf._mtiles(Q.shape[0])
    F = torch.zeros(2 * 16 * MT * D, dtype=torch.float16, device='cuda')
    t = torch.full((1,), t0, dtype=torch.int32, device='cuda')
    blocks = B * H * -(-P // (16 if kernel == 'pf_attn16' else 64))
    e._plan = []
    p, i = pf._p, pf._i
    e._launch(kernel, 8 * -(-blocks // 8), [p(Q), p(k), p(v), i(B), i(P), p(t), i(1), i(L), i(TMAX), i(H), p(F), i(MT),
                                            p(e.err)])
    plan, e._plan = e._plan, []
    e._replay(plan)
    torch.cuda.synchronize()
    hi, lo = F.view(2, MT, D // 32, 4, 16, 8).permute(0, 1, 4, 2, 3, 5).reshape(2, -1, D).double()
    return (hi + lo / 2048)[:M].view(B, P, H, 64)


def _inputs(P, t0, scale=1.0):
    import torch
    gen = torch.Generator(device='cuda').manual_seed(1000 * P + t0)
    Q = torch.randn(B * P, D, generator=gen, device='cuda') * scale
    k, v = (torch.randn(B, L, TMAX, H, 64, generator=gen, device='cuda').half() for _ in range(2))
    return Q, k, v


def _check(got, Q, k, v, t0, P):
    """Against 64 bits. A score's error is that of 22-bit queries and 64 fp32 additions, relative to the sum of its
    terms' magnitudes; the output's is twice the largest score error (numerator and sum), the 22-bit weights and n fp32
    additions of each, relative to the largest value."""
    import torch
    q = Q.view(B, P, H, 64).double().permute(0, 2, 1, 3)
    n = t0 + P
    K, V = (c[:, 1, :n].double().permute(0, 2, 1, 3) for c in (k, v))
    s = q @ K.transpose(2, 3).contiguous() / 8
    later = torch.ones(P, n, dtype=torch.bool, device='cuda').triu(t0 + 1)
    s = s.masked_fill(later, -torch.inf)
    want = (torch.softmax(s, -1) @ V).permute(0, 2, 1, 3)
    ds = (q.abs() @ K.nan_to_num(0, 0, 0).abs().transpose(2, 3).contiguous()).max().item() / 8 * (2.0 ** -22 + 2.0 ** -18)
    bound = V.abs().max().item() * (2 * ds + 2.0 ** -21 + 2 * n * 2.0 ** -24)
    assert (got - want).abs().max().item() <= bound


@pytest.mark.parametrize('kernel', ['pf_attn', 'pf_attn16'])
@pytest.mark.parametrize('P', [2, 8, 15, 16, 17, 63, 64, 65, 130])
def test_prefill_attention_matches_64_bits(engine, kernel, P):
    for t0 in (0, 1, 62, 64, 200):
        Q, k, v = _inputs(P, t0)
        k[:, :, t0 + P:], v[:, :, t0 + P:] = float('nan'), float('inf')      # rows no query may see
        _check(_run(engine, kernel, Q, k, v, t0, P), Q, k, v, t0, P)
    engine.check()


@pytest.mark.parametrize('kernel', ['pf_attn', 'pf_attn16'])
def test_prefill_attention_takes_any_query_magnitude(engine, kernel):
    import torch
    P, t0 = 20, 70
    for scale in (1e-30, 1e-6, 1e-3):
        Q, k, v = _inputs(P, t0, scale)
        _check(_run(engine, kernel, Q, k, v, t0, P), Q, k, v, t0, P)
    # far beyond the fp16 range: the softmax is one position's
    Q, k, v = _inputs(P, t0, 1e6)
    got = _run(engine, kernel, Q, k, v, t0, P)
    q0 = Q.view(B, P, H, 64)[:, 0].double()                                        # the first query of each row
    best = torch.einsum('bhd,bshd->bhs', q0.cpu(), k[:, 1, :t0 + 1].double().cpu()).argmax(-1)
    for b in range(B):
        for h in range(H):
            assert (got[b, 0, h] - v[b, 1, best[b, h], h].double()).abs().max().item() < 1e-5
    engine.check()


@pytest.mark.parametrize('kernel', ['pf_attn', 'pf_attn16'])
@pytest.mark.parametrize('q7', [-0.5, -0.3, -1e-9, -1e-30])
def test_a_key_of_minus_infinite_score_has_no_weight(engine, kernel, q7):
    """A cache row that overflowed fp16 in one key component: queries whose score there is -inf ignore it, whichever of
    their component's planes are 0 (-0.5: all but the first; below 2^-25 of the largest: the first)."""
    P, t0 = 5, 90
    Q, k, v = _inputs(P, t0)
    Q.view(B, P, H, 64)[..., 7] = q7
    k[:, 1, 40, :, 7] = float('inf')
    _check(_run(engine, kernel, Q, k, v, t0, P), Q, k, v, t0, P)
    engine.check()


@pytest.mark.parametrize('kernel', ['pf_attn', 'pf_attn16'])
@pytest.mark.parametrize('q7', [0.5, 1e-9, 0.0])
def test_an_infinite_or_undefined_score_is_refused(engine, kernel, q7):
    """+inf (its weight is inf - inf) and 0 * inf: the outputs are no numbers, and the range word says so."""
    P, t0 = 5, 90
    Q, k, v = _inputs(P, t0)
    Q.view(B, P, H, 64)[..., 7] = q7
    k[:, 1, 40, :, 7] = float('inf')
    assert _run(engine, kernel, Q, k, v, t0, P).isnan().all()
    with pytest.raises(RuntimeError, match='fp16 range'):
        engine.check()


def _in_fp32(Q, k, v, t0, P):
    """The attention with every operation in fp32 (each rounded from 64 bits here): eight lanes of 8 dims a dot, added
    pairwise, exponentials and their sum over 64 lanes, weights divided by it, values in 8 residues of the positions."""
    import torch

    def pairwise(x):                                            # over the first axis, a power of two long
        while x.shape[0] > 1:
            x = x[0::2] + x[1::2]
        return x[0]

    def fma(a, b, c):
        return (a.double() * b.double() + c.double()).float()

    n = t0 + P
    q = Q.view(B, P, H, 1, 8, 8).float()
    K, V = (c[:, 1, :n].permute(0, 2, 1, 3).float() for c in (k, v))        # [B, H, n, 64]
    acc = torch.zeros(B, P, H, n, 8, device='cuda')
    for j in range(8):
        acc = fma(q[..., j], K.view(B, 1, H, n, 8, 8)[..., j], acc)
    s = pairwise(acc.movedim(-1, 0)) * 0.125
    seen = torch.arange(n, device='cuda') <= t0 + torch.arange(P, device='cuda')[:, None, None]
    s = s.masked_fill(~seen, -torch.inf)
    ex = (s - s.amax(-1, keepdim=True)).double().exp().float()
    lanes = torch.zeros(B, P, H, 64 * -(-n // 64), device='cuda')
    lanes[..., :n] = ex
    total = torch.zeros(B, P, H, 64, device='cuda')
    for part in lanes.split(64, -1):
        total = total + part
    w = ex / pairwise(total.movedim(-1, 0))[..., None]
    out = torch.zeros(8, B, P, H, 64, device='cuda')
    for i in range(n):
        out[i % 8] = fma(w[..., i, None], V[:, None, :, i], out[i % 8])
    return pairwise(out)


@pytest.mark.parametrize('kernel', ['pf_attn', 'pf_attn16'])
@pytest.mark.parametrize('P,t0', [(37, 0), (130, 0), (130, 100), (128, 200), (20, 310)])
def test_prefill_attention_is_as_exact_as_fp32(engine, kernel, P, t0):
    """No further from 64 bits (2-norm) than fp32 arithmetic throughout, for queries, keys and values at the scale GPT-2
    small's projections give. Both distances are root mean squares over N = B P H 64 >= 7680 values, each known to
    1 / sqrt(2 N) = 0.8% of itself: 3% of their quotient is more than twice that of both."""
    import torch
    Q, k, v = _inputs(P, t0, 0.55)
    k, v = ((0.55 * c.float()).half() for c in (k, v))
    q = Q.view(B, P, H, 64).double().permute(0, 2, 1, 3)
    K, V = (c[:, 1, :t0 + P].double().permute(0, 2, 1, 3) for c in (k, v))
    s = (q @ K.transpose(2, 3).contiguous() / 8).masked_fill(
        torch.ones(P, t0 + P, dtype=torch.bool, device='cuda').triu(t0 + 1), -torch.inf)
    want = (torch.softmax(s, -1) @ V).permute(0, 2, 1, 3)
    plain = _in_fp32(Q, k, v, t0, P)
    hi = plain.half()
    plain = hi.double() + ((plain - hi.float()) * 2048).half().double() / 2048      # as the next product reads it
    off, off32 = ((x - want).norm().item() for x in (_run(engine, kernel, Q, k, v, t0, P), plain))
    print(f'{kernel} {P} after {t0}: {off / want.norm().item():.3e}, in fp32 {off32 / want.norm().item():.3e}')
    assert off <= 1.03 * off32
    engine.check()
