"""The products beyond 64 rows (hip/prefill.hip pf_pgemm*) on the GPU, each
output tile forced in turn, against plain PyTorch in 64 bits: rows and
columns at and around the edges of the tiles, each epilogue, split folds; and
the LayerNorms of many rows."""
import pytest

pytestmark = pytest.mark.gpu

D, F, TMAX = 192, 768, 300


@pytest.fixture(scope='module')
def engine():
    import torch
    if not torch.cuda.is_available():
        pytest.skip('no GPU')
    from vesta.gpt2 import VestaGPT2
    from vesta.weights import GPT2Shape, RandomGPT2
    return VestaGPT2(RandomGPT2(GPT2Shape(2, D, 3, F, vocab=203), 5), batch=1, tmax=TMAX, engine='layered')


def _frag(A):
    """Activations [M, K] in fragment order (hi and lo planes) as the kernels' producers write them."""
    import torch
    from vesta.prefill import _mtiles, frag_weights
    M, K = A.shape
    A = torch.cat([A, A.new_zeros(16 * _mtiles(M) - M, K)])
    hi = A.half()
    return torch.stack([frag_weights(hi), frag_weights(((A - hi.float()) * 2048).half())]).contiguous()


def _unfrag(f, M, K):
    import torch
    from vesta.prefill import _mtiles
    hi, lo = f.view(2, _mtiles(M), K // 32, 4, 16, 8).permute(0, 1, 4, 2, 3, 5).reshape(2, -1, K).double()
    return (hi + lo / 2048)[:M]


def _close(got, want, bound):
    """|got - want| within ``bound`` (the largest error the arithmetic allows, per element)."""
    over = ((got.double() - want).abs() / bound).max().item()
    assert over <= 1, over


def _exact(W, a, name, layer):
    """The product, and its bound: 22-bit activations (2^-22 each) and K fp32 additions (2^-24 each) of terms whose
    absolute values sum to s; plus rounding of the epilogue's few fp32 operations."""
    w = W[name][layer].double()
    s = a.double().abs() @ w.abs()
    return a.double() @ w, s * (2.0 ** -22 + a.shape[1] * 2.0 ** -24)


def _gelu(u):
    """GELU in 64 bits, and its error per error of u (its slope is below 1.13; its exponential is good to 2^-20)."""
    import torch
    return 0.5 * u * (1 + torch.tanh(0.7978845608028654 * (u + 0.044715 * u ** 3))), 2.0 ** -20 * (u.abs() + 2.0 ** -10)


def _check_cache(m, layer, t0, rows, P, want, bound):
    """The cache rows of ``rows`` x P positions from t0 in fp16; those at or past the end are dropped, all others zero."""
    import torch
    n = max(0, min(P, m.tmax - t0))
    for part, cache in ((1, m.keys), (2, m.vals)):
        c = slice(part * D, (part + 1) * D)
        w, b = (x.view(rows, P, -1)[:, :n, c] for x in (want, bound))
        _close(cache[:rows, layer, t0:t0 + n].reshape(rows, n, D), w, b + 2.0 ** -11 * w.abs() + 2.0 ** -25)
        rest = cache.clone()
        rest[:rows, layer, t0:t0 + n] = 0
        assert not rest.any()


@pytest.mark.parametrize('kernel', ['pf_pgemm128', 'pf_pgemm64', 'pf_pgemm64w', 'pf_pgemm32'])
@pytest.mark.parametrize('M', [65, 127, 128, 129, 257])
def test_products_match_64_bits(engine, monkeypatch, kernel, M):
    import torch
    from vesta import prefill as pf
    m, e, layer, P = engine, engine._pf, 1, M
    W = m.W
    gen = torch.Generator(device='cuda').manual_seed(M)
    A, G, Z = (torch.randn(M, n, generator=gen, device='cuda') for n in (D, F, D))

    def plan(ks):
        monkeypatch.setattr(pf, 'pgemm_plan', lambda *a: (kernel, ks))
        e._plan = []
        e._ws = None

    def run():
        p, e._plan = e._plan, []
        e._replay(p)
        torch.cuda.synchronize()
        e.check()

    def exact(a, name):
        return _exact(W, a, name, layer)

    bias = {n: W[n][layer].double() for n in ('qkvb', 'ob', 'fcb', 'pb')}
    # qkv: queries in fp32, cache rows in fp16, all of them inside the cache and some past its end
    for t0 in (7, TMAX - 60):
        plan(1)
        m.seek(t0)
        m.keys.zero_(), m.vals.zero_()
        Q = torch.empty(M, D, device='cuda')
        e._pgemm(_frag(A), D, 'qkvw', layer, 3 * D, pf.MODE_QKV, bias=W['qkvb'][layer], out=Q, ldo=D, M=M, P=P)
        run()
        want, bound = exact(A, 'qkvw')
        want, bound = want + bias['qkvb'], bound + 2.0 ** -23 * (want.abs() + 1)
        _close(Q, want[:, :D], bound[:, :D])
        _check_cache(m, layer, t0, 1, P, want, bound)
    # GELU in fragment order (another 22-bit rounding)
    plan(1)
    out = torch.zeros(2 * 16 * pf._mtiles(M) * F, dtype=torch.float16, device='cuda')
    e._pgemm(_frag(A), D, 'fcw', layer, F, pf.MODE_GELU, bias=W['fcb'][layer], F=out, M=M)
    run()
    want, bound = exact(A, 'fcw')
    want, own = _gelu(want + bias['fcb'])
    _close(_unfrag(out, M, F), want, 1.13 * bound + own)
    # residual, whole and with a split fold whose parts the next LayerNorm's launch adds
    want, bound = exact(G, 'pw')
    want, bound = want + bias['pb'] + Z.double(), bound + 2.0 ** -22 * (want.abs() + Z.double().abs() + 1)
    for ks in (1, 2, 3):
        plan(ks)
        z = Z.clone()
        nf = torch.zeros(2 * 16 * pf._mtiles(M) * D, dtype=torch.float16, device='cuda')
        done = e._pgemm(_frag(G), F, 'pw', layer, D, pf.MODE_RESID, bias=W['pb'][layer], out=z, ldo=D,
                        ln=(W['ln1w'][layer], W['ln1b'][layer], nf), M=M)
        assert done == (ks > 1)
        run()
        _close(z, want, bound)
        if done:
            c = z.double() - z.double().mean(-1, keepdim=True)
            y = c / torch.sqrt((c * c).mean(-1, keepdim=True) + 1e-5)      # gains 1, biases 0
            _close(_unfrag(nf, M, D), y, 2.0 ** -18 * (y.abs() + 1))
    # plain, with a column count no tile divides (the output head)
    plan(1)
    V = W['wte'].shape[0]
    out = torch.zeros(M, V, device='cuda')
    e._pgemm(_frag(A), D, 'wte', None, V, pf.MODE_PLAIN, out=out, ldo=V, M=M)
    run()
    w = W['wte'].double()
    _close(out, A.double() @ w.t(), (A.double().abs() @ w.abs().t()) * (2.0 ** -22 + D * 2.0 ** -24))


@pytest.fixture(scope='module')
def engine3():
    """Three batch rows, 24 layers: prompts of 2 to 8 tokens keep their order of sums."""
    import torch
    if not torch.cuda.is_available():
        pytest.skip('no GPU')
    from vesta.gpt2 import VestaGPT2
    from vesta.weights import GPT2Shape, RandomGPT2
    return VestaGPT2(RandomGPT2(GPT2Shape(24, D, 3, F, vocab=203), 7), batch=3, tmax=TMAX, engine='layered')


@pytest.mark.parametrize('kernel,P,t0', [
    (k, P, t0) for k in ('pf_mgemm', 'pf_pgemm128', 'pf_pgemm64', 'pf_pgemm64w', 'pf_pgemm32', 'pf_pgemm32o')
    for P, t0 in ((2, 5), (5, 298), (7, 0), (19, 290), (21, 40), (43, 270), (101, 3)) if k != 'pf_mgemm' or 3 * P <= 64])
def test_new_cache_rows_go_to_their_batch_row_and_position(engine3, monkeypatch, kernel, P, t0):
    """Three rows of prompt lengths that no tile divides, in tiled products of few rows too, whole and (pf_pgemm32o) with
    the fold in parts that pf_reduce adds."""
    import torch
    from vesta import prefill as pf
    m, M, layer = engine3, 3 * P, 5
    e, W = m._pf, m.W
    gen = torch.Generator(device='cuda').manual_seed(P)
    A = torch.randn(M, D, generator=gen, device='cuda')
    monkeypatch.setattr(pf, 'pgemm_plan', lambda *a: (kernel, 1))
    want, bound = _exact(W, A, 'qkvw', layer)
    want, bound = want + W['qkvb'][layer].double(), bound + 2.0 ** -23 * (want.abs() + 1)
    for ks in (1, 2, 3) if kernel == 'pf_pgemm32o' else (None,):
        m.seek(t0)
        m.keys.zero_(), m.vals.zero_()
        Q = torch.empty(M, D, device='cuda')
        e._plan = []
        kw = dict(bias=W['qkvb'][layer], out=Q, ldo=D, M=M, P=P)
        if kernel == 'pf_mgemm':
            e._mgemm(_frag(A), D, 'qkvw', layer, 3 * D, pf.MODE_QKV, **kw)
        else:
            e._pgemm(_frag(A), D, 'qkvw', layer, 3 * D, pf.MODE_QKV, ks=ks, **kw)
        plan, e._plan = e._plan, []
        assert plan[0][0].startswith(kernel)
        e._replay(plan)
        e.check()
        _close(Q, want[:, :D], bound[:, :D])
        _check_cache(m, layer, t0, 3, P, want, bound)


@pytest.mark.parametrize('M', [2, 8, 17, 33, 64, 130])
def test_ordered_products_match_64_bits(engine, M):
    """pf_pgemm32o at few rows, where it clamps its row tiles, its fold whole and in parts: GELU (parts added by
    pf_reduce_frag), and the residual with the LayerNorm after it and without (pf_reduce_ln, pf_reduce)."""
    import torch
    from vesta import prefill as pf
    m, e, layer = engine, engine._pf, 1
    W = m.W
    gen = torch.Generator(device='cuda').manual_seed(M)
    A, G, Z = (torch.randn(M, n, generator=gen, device='cuda') for n in (D, F, D))

    def run():
        p, e._plan = e._plan, []
        e._replay(p)
        e.check()

    for ks in (1, 2, 3):
        out = torch.zeros(2 * 16 * pf._mtiles(M) * F, dtype=torch.float16, device='cuda')
        e._plan = []
        e._pgemm(_frag(A), D, 'fcw', layer, F, pf.MODE_GELU, bias=W['fcb'][layer], F=out, M=M, ks=ks)
        run()
        want, bound = _exact(W, A, 'fcw', layer)
        want, own = _gelu(want + W['fcb'][layer].double())
        _close(_unfrag(out, M, F), want, 1.13 * bound + own)
        want, bound = _exact(W, G, 'pw', layer)
        want, bound = want + W['pb'][layer].double() + Z.double(), bound + 2.0 ** -22 * (want.abs() + Z.double().abs() + 1)
        for norm in (False, True):
            z, nf = Z.clone(), torch.zeros(2 * 16 * pf._mtiles(M) * D, dtype=torch.float16, device='cuda')
            done = e._pgemm(_frag(G), F, 'pw', layer, D, pf.MODE_RESID, bias=W['pb'][layer], out=z, ldo=D,
                            ln=(W['ln1w'][layer], W['ln1b'][layer], nf) if norm else None, M=M, ks=ks)
            run()
            assert done == (norm and ks > 1)
            _close(z, want, bound)
            if done:
                c = z.double() - z.double().mean(-1, keepdim=True)
                y = c / torch.sqrt((c * c).mean(-1, keepdim=True) + 1e-5)      # gains 1, biases 0
                _close(_unfrag(nf, M, D), y, 2.0 ** -18 * (y.abs() + 1))


@pytest.mark.parametrize('P', [2, 5, 8, 9])
@pytest.mark.parametrize('t0', [0, 6])
def test_short_prompts_of_a_deep_model_match_single_steps(engine3, P, t0):
    """24 layers, from an empty cache (up to 8 tokens: in the kept order of sums) and continued, against the same tokens
    one decode step each: the same logits within the engines' tolerance, the same cache rows within fp16's rounding and
    what it carries on (2^-9 of the largest value)."""
    import torch
    from vesta import prefill as pf
    from vesta.weights import random_prompts
    m = engine3
    assert pf.ordered(P, m.L, t0) == (t0 == 0 and P <= 8)
    pr = torch.from_numpy(random_prompts(3, 6 + P, 203, seed=P)).to('cuda', torch.int32)
    got = []
    for mode in ('batched', 'steps'):
        m.reset()
        if t0:
            m.prefill(pr[:, :t0].contiguous(), mode='steps')
        m.prefill(pr[:, t0:t0 + P].contiguous(), mode=mode)
        m.check()
        assert int(m.t) == t0 + P
        got.append([x.float().clone() for x in (m.logits(), m.keys, m.vals)] + [m.x.clone()])
    (lb, kb, vb, xb), (ls, ks, vs, xs) = got
    assert (lb - ls).abs().max() < 1e-3
    for a, b in ((kb, ks), (vb, vs)):
        assert (a - b).abs().max() <= 2.0 ** -9 * b.abs().max()
    top = ls.topk(2, -1).values
    clear = top[:, 0] - top[:, 1] > 2e-3
    assert clear.any() and torch.equal(xb[clear], xs[clear])


@pytest.mark.parametrize('K,apart', [(1024, 1.57), (3072, 2.34)])
def test_a_long_fold_is_nearly_as_exact_as_a_short_one(engine, monkeypatch, K, apart):
    """pf_pgemm32, which takes long folds whole at some hundred rows, sums 128 of them at a time. In rounding units, with
    partial sums that grow as the square root of their length, c sums of s k-steps added in order are
    (s + 1) / 2 - 1 / s + (c + 1) / 2 - 1 / c squared from 64 bits, relative to the result, plus what a k-step's own sums
    leave; so with s = 4 a fold of 1024 is at most sqrt(6.6 / 3.25) = 1.43 times as far as one of 256, one of 3072 2.13
    times (one running sum: measured 1.73 and 2.9). 10% for the samples and the model."""
    import torch
    from vesta import prefill as pf
    m, e, M, N = engine, engine._pf, 129, 768
    monkeypatch.setattr(pf, 'pgemm_plan', lambda *a: ('pf_pgemm32', 1))
    off = []
    for k in (256, K):
        gen = torch.Generator(device='cuda').manual_seed(k)
        A, w = (torch.randn(*s, generator=gen, device='cuda') for s in ((M, k), (N, k)))
        w = (0.02 * w).half()
        Wf = pf.frag_weights(w).contiguous()
        monkeypatch.setattr(e, '_frag', lambda name: Wf)
        out, F = torch.zeros(M, N, device='cuda'), _frag(A)
        e._plan = []
        e._pgemm(F, k, 'w', None, N, pf.MODE_PLAIN, out=out, ldo=N, M=M)
        plan, e._plan = e._plan, []
        e._replay(plan)
        want = _unfrag(F, M, k) @ w.double().t()
        off.append(((out.double() - want).norm() / want.norm()).item())
    print(f'{K}: {off[1]:.3e}, 256: {off[0]:.3e}')
    assert off[1] <= apart * off[0]
    e.check()


def test_more_than_64_rows_decode_and_prefill_like_fewer():
    """70 rows (products in output tiles, the output head too) against the same rows in a batch of 7, whose prompt goes a
    step at a time (products of few rows): the same tokens where the margin is clear, logits within the engines'
    tolerance."""
    import torch
    from vesta.gpt2 import VestaGPT2
    from vesta.weights import GPT2Shape, RandomGPT2, random_prompts
    hf = RandomGPT2(GPT2Shape(2, D, 3, F, vocab=203), 5)
    pr = torch.from_numpy(random_prompts(70, 9, 203, seed=3)).to('cuda', torch.int32)
    seven = torch.arange(0, 70, 10, device='cuda') + 9
    got = []
    for rows in (torch.arange(70, device='cuda'), seven):
        n = len(rows)
        mine = slice(None) if n == 7 else seven
        m = VestaGPT2(hf, batch=n, tmax=32, engine='layered')
        m.reset()
        m.prefill(pr[rows].contiguous(), mode='batched' if n == 70 else 'steps')
        lg, tok = [m.logits()[mine].clone()], [m.x[mine].clone()]
        for _ in range(3):
            m.x.copy_(pr[rows, 0])
            m.step()
            lg.append(m.logits()[mine].clone())
            tok.append(m.x[mine].clone())
        m.check()
        got.append((torch.stack(lg), torch.stack(tok)))
    (l70, t70), (l7, t7) = got
    assert (l70 - l7).abs().max() < 1e-3
    top = l7.topk(2, -1).values
    clear = top[..., 0] - top[..., 1] > 2e-3
    assert clear.sum() > 20 and torch.equal(t70[clear], t7[clear])


@pytest.mark.parametrize('D', [64, 1024, 1088, 2048])
@pytest.mark.parametrize('M', [1, 17, 48])
def test_layer_norm_of_sixteen_rows_a_block_matches_64_bits(engine, D, M):
    """pf_lnm*: widths at the ends of each kernel's range, rows around a block's 16."""
    import torch
    from vesta import prefill as pf
    e = engine._pf
    gen = torch.Generator(device='cuda').manual_seed(D + M)
    X, w, b = (torch.randn(*s, generator=gen, device='cuda') for s in ((M, D), (D,), (D,)))
    w, b = w.half(), b.half()
    F = torch.zeros(2 * 16 * pf._mtiles(M) * D, dtype=torch.float16, device='cuda')
    e._plan = []
    p, i = pf._p, pf._i
    e._launch('pf_lnm8' if D <= 1024 else 'pf_lnm16', -(-M // 16), [p(X), i(M), i(D), p(w), p(b), p(F),
                                                                     i(pf._mtiles(M)), p(e.err)])
    plan, e._plan = e._plan, []
    e._replay(plan)
    x = X.double()
    c = x - x.mean(-1, keepdim=True)
    y = c / torch.sqrt((c * c).mean(-1, keepdim=True) + 1e-5)
    want = y * w.double() + b.double()
    # sums of D fp32 terms (2^-24 each, at most sqrt(D) long along a lane, lanes and waves), four roundings, 22 bits
    _close(_unfrag(F, M, D), want, (2.0 ** -21 + D ** 0.5 * 2.0 ** -24) * ((y * w.double()).abs() + b.double().abs() + 1))
    e.check()


@pytest.mark.parametrize('shape', [(2, 192, 3, 768), (1, 1600, 25, 6400)])
def test_up_to_eight_rows_compute_what_more_rows_compute(shape):
    """Products of at most 8 rows hold both halves of the activations in one operand tile; each row's sums are those of
    the same rows in a batch of 9, bit for bit (the wider shape: waves with more k-steps than one batch of loads)."""
    import torch
    from vesta.gpt2 import VestaGPT2
    from vesta.weights import GPT2Shape, RandomGPT2, random_prompts
    hf = RandomGPT2(GPT2Shape(*shape, vocab=203), 6)
    pr = torch.from_numpy(random_prompts(9, 4, 203, seed=4)).to('cuda', torch.int32)
    got = []
    for rows in (9, 8, 3, 1):
        m = VestaGPT2(hf, batch=rows, tmax=16, engine='layered')
        m.reset()
        for k in range(4):
            m.x.copy_(pr[:rows, k])
            m.step()
        m.check()
        got.append((m.logits().clone(), m.keys.clone(), m.vals.clone()))
    for rows, g in zip((8, 3, 1), got[1:]):
        for a, b in zip(g, got[0]):
            assert torch.equal(a, b[:rows])


def _lnm_and_ln(e, X, w, b):
    """The LayerNorm of X's rows by a block per 16 rows and by a block per row, as fp32 pairs of planes."""
    import torch
    from vesta import prefill as pf
    M, D = X.shape
    p, i, MT = pf._p, pf._i, pf._mtiles(M)
    out = []
    for name in ('pf_lnm8' if D <= 1024 else 'pf_lnm16', 'pf_ln'):
        F = torch.zeros(2 * 16 * MT * D, dtype=torch.float16, device='cuda')
        e._plan = []
        if name == 'pf_ln':
            e._launch(name, M, [p(X), i(0), i(1), p(w), p(b), i(D), p(F), i(MT), p(e.err)])
        else:
            e._launch(name, -(-M // 16), [p(X), i(M), i(D), p(w), p(b), p(F), i(MT), p(e.err)])
        plan, e._plan = e._plan, []
        e._replay(plan)
        out.append(_unfrag(F, M, D))
    return out


@pytest.mark.parametrize('D', [768, 1024, 1600, 2048])
@pytest.mark.parametrize('mean', [0.0, 30.0])
def test_layer_norm_of_many_rows_is_as_exact_as_of_few(engine, D, mean):
    """Both kernels' distances from 64 bits (2-norm) over 999 rows. Distances are over 999 * D values, but the error of a
    row's mean is common to its D values: 999 samples of each, 2.2% of a root mean square, 3.2% of the quotient of two,
    10% three times that."""
    import torch
    gen = torch.Generator(device='cuda').manual_seed(D)
    X, w, b = (torch.randn(*s, generator=gen, device='cuda') for s in ((999, D), (D,), (D,)))
    X, w, b = X + mean, (1 + 0.1 * w).half(), (0.02 * b).half()
    c = X.double() - X.double().mean(-1, keepdim=True)
    want = c / torch.sqrt((c * c).mean(-1, keepdim=True) + 1e-5) * w.double() + b.double()
    many, few = ((y - want).norm().item() for y in _lnm_and_ln(engine._pf, X, w, b))
    print(f'{D} wide, mean {mean}: {many / want.norm().item():.3e}, a block per row {few / want.norm().item():.3e}')
    assert many <= 1.1 * few
    engine.check()


@pytest.mark.parametrize('D', [768, 1600, 2048])
@pytest.mark.parametrize('size', [1e15, 1e18, 4e18, 1e20, 1e30])
def test_layer_norm_of_many_rows_takes_what_of_few_takes(engine, D, size):
    """Rows whose squares reach, and pass, the end of fp32's range: what a block per row accepts (its biases, where the
    variance is infinite) a block per 16 rows accepts, with the same result to their sums' rounding."""
    import torch
    gen = torch.Generator(device='cuda').manual_seed(D)
    X, w, b = (torch.randn(*s, generator=gen, device='cuda') for s in ((33, D), (D,), (D,)))
    X[::2] = X[::2] * size                                       # large rows beside small ones
    X[6, 1:] = 0                                                 # one value alone
    many, few = _lnm_and_ln(engine._pf, X, w.half(), b.half())
    engine.check()
    _close(many, few, (2.0 ** -20 + D ** 0.5 * 2.0 ** -23) * (many.abs() + few.abs() + 1))


def test_a_prompt_of_many_rows_matches_its_rows_alone():
    """1600 rows of activations (LayerNorms of 16 rows a block, from the batched pass itself) against two of its batch
    rows in a model of their own, 400 rows (a block per row): the same cache rows within fp16's rounding and what it
    carries on (2^-9 of the largest value), logits within the engines' tolerance."""
    import torch
    from vesta import prefill as pf
    from vesta.gpt2 import VestaGPT2
    from vesta.weights import GPT2Shape, RandomGPT2, random_prompts
    hf = RandomGPT2(GPT2Shape(2, D, 3, F, vocab=203), 8)
    pr = torch.from_numpy(random_prompts(8, 200, 203, seed=9)).to('cuda', torch.int32)
    got = []
    for rows in ([0, 1, 2, 3, 4, 5, 6, 7], [2, 7]):
        m = VestaGPT2(hf, batch=len(rows), tmax=208, engine='layered')
        m.prefill(pr[rows].contiguous())
        m.check()
        names = {x[0] for x in m._pf._plans[200, False]}
        assert ('pf_lnm8' in names) == (len(rows) * 200 >= pf.LNM_ROWS)
        mine = [2, 7] if len(rows) == 8 else [0, 1]
        got.append([x[mine].float() for x in (m.logits(), m.keys, m.vals)])
    assert (got[0][0] - got[1][0]).abs().max() < 1e-3
    for a, b in zip(got[0][1:], got[1][1:]):
        assert (a - b).abs().max() <= 2.0 ** -9 * b.abs().max()
