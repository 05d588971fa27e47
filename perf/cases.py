"""The work a program using this package has it do, as cases that can be timed and compared.

A case is one call of ``VestaGPT2`` with what a serving program does around it:

* ``kind='decode'``: rows that already hold ``pos`` tokens are set to that
  position, given their next token and advanced ``steps`` greedy steps in one
  ``step()`` call. Results: the tokens chosen at each step, the last step's
  logits and the key / value cache rows the steps wrote.
* ``kind='prefill'``: ``prompt`` new tokens per row are fed at position
  ``pos`` (0: a fresh sequence; above: a conversation continued) in one
  ``prefill()`` call. Results: the token chosen after the prompt, its logits
  and the cache rows written.

The models are the three sizes the package carries programs for, at random
initialisation: the weights N(0, 0.02) of the architecture's own
initialisation, LayerNorm gains around 1 and small biases; the cache rows
already there are drawn at the scale the key and value projections give.
"""
import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / 'vesta-gpu_amd'))

from vesta.gpt2 import VestaGPT2  # noqa: E402
from vesta.weights import SHAPES, layer_tensors  # noqa: E402


def _case(name, kind, model, rows, pos, tmax, steps=0, prompt=0):
    return dict(name=name, kind=kind, model=model, rows=rows, pos=pos, tmax=tmax, steps=steps, prompt=prompt)


def listed():
    return [
        # one sequence, one step per call: a program that looks at each token before it goes on
        # (the benchmark's one-launch-per-step protocol); the smallest call, latency alone
        _case('decode_small_b1', 'decode', 'small', 1, 256, 448, steps=1),
        # the benchmark's own workload: 8 rows at its mean context, many steps per call
        _case('decode_small_b8', 'decode', 'small', 8, 248, 448, steps=16),
        # a batch of a size no tile is made for, after short prompts
        _case('decode_small_b13', 'decode', 'small', 13, 61, 448, steps=4),
        # a server's batch late in long conversations: the cache rows are most of the bytes
        _case('decode_small_b32', 'decode', 'small', 32, 892, 1024, steps=4),
        # the middle size at the benchmark's batch, two thirds into its cache
        _case('decode_medium_b8', 'decode', 'medium', 8, 384, 512, steps=8),
        # one user of the largest model
        _case('decode_xl_b1', 'decode', 'xl', 1, 200, 512, steps=4),
        # the largest model at the largest batch
        _case('decode_xl_b64', 'decode', 'xl', 64, 190, 256, steps=2),
        # a short question: the time to the first token
        _case('prefill_small_1x37', 'prefill', 'small', 1, 0, 448, prompt=37),
        # the benchmark's prompts
        _case('prefill_small_8x128', 'prefill', 'small', 8, 0, 448, prompt=128),
        # long documents for a server's whole batch
        _case('prefill_small_32x768', 'prefill', 'small', 32, 0, 1024, prompt=768),
        # three conversations continued by a ragged number of tokens
        _case('prefill_medium_3x333', 'prefill', 'medium', 3, 100, 512, prompt=333),
        # the largest model's prompts at its largest batch
        _case('prefill_xl_64x128', 'prefill', 'xl', 64, 0, 256, prompt=128),
    ]


# what draw() may take of each model: the most rows of a decode step, the most prompt tokens of a
# prefill over all rows (so that no drawn case costs more than the largest listed one), cache lengths
_RANGE = {'small': (64, 24576, (128, 256, 448, 512, 777, 1024)),
          'medium': (32, 12288, (128, 256, 512, 600)),
          'xl': (64, 7168, (128, 256, 512))}


def _spread(rng, low, high):
    """A whole number from low to high, spread over its logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(('decode', 'prefill'))
    model = rng.choice(('small', 'small', 'medium', 'xl'))
    rows_max, tokens_max, tmaxes = _RANGE[model]
    tmax = rng.choice(tmaxes)
    if kind == 'decode':
        steps = _spread(rng, 1, 16 if model == 'small' else 4)
        return dict(kind=kind, model=model, rows=_spread(rng, 1, rows_max), pos=rng.randrange(1, tmax - steps),
                    tmax=tmax, steps=steps, prompt=0)
    prompt = _spread(rng, 3, tmax - 1)
    rows = _spread(rng, 1, max(1, min(64, tokens_max // prompt)))
    pos = 0 if rng.random() < 0.6 else rng.randrange(0, tmax - prompt)
    return dict(kind=kind, model=model, rows=rows, pos=pos, tmax=tmax, steps=0, prompt=prompt)


class _Weights:
    """Seeded fp16 weights under Hugging Face names, made on the device."""

    def __init__(self, model, gen):
        cfg = self.config = SHAPES[model]

        def normal(shape, std=0.02, mean=0.0):
            return (torch.randn(shape, generator=gen, device='cuda') * std + mean).half()

        def layer_norm(name, shape):
            return normal(shape, 0.1, 1.0) if name.endswith('weight') else normal(shape)

        sd = {'transformer.wte.weight': normal((cfg.vocab, cfg.n_embd)),
              'transformer.wpe.weight': normal((cfg.n_positions, cfg.n_embd))}
        for i in range(cfg.n_layer):
            for name, shape, is_norm in layer_tensors(cfg):
                sd[f'transformer.h.{i}.{name}'] = layer_norm(name, shape) if is_norm else normal(shape)
        for name in ('ln_f.weight', 'ln_f.bias'):
            sd['transformer.' + name] = layer_norm(name, (cfg.n_embd,))
        self._sd = sd

    def state_dict(self):
        return self._sd


def _inputs(case, seed):
    """Weights, the new tokens [rows, 1 or prompt] and the cache rows before ``pos`` (keys and values,
    [rows, layers, pos, heads, 64]), from the seed alone."""
    gen = torch.Generator(device='cuda').manual_seed(int(seed) * 2 + 1)
    weights = _Weights(case['model'], gen)
    cfg = weights.config
    tokens = torch.randint(0, cfg.vocab, (case['rows'], case['prompt'] or 1), generator=gen, device='cuda',
                           dtype=torch.int32)
    scale = 0.02 * math.sqrt(cfg.n_embd)
    past = [torch.randn((case['rows'], cfg.n_layer, case['pos'], cfg.n_head, cfg.head_dim), generator=gen,
                        device='cuda', dtype=torch.float16) * scale for _ in range(2)]
    return weights, tokens, past


def prepare(case, seed):
    weights, tokens, past = _inputs(case, seed)
    m = VestaGPT2(weights, batch=case['rows'], tmax=case['tmax'])
    m.keys[:, :, :case['pos']] = past[0]
    m.vals[:, :, :case['pos']] = past[1]
    state = dict(m=m, tokens=tokens, pos=case['pos'], steps=case['steps'], prompt=case['prompt'])
    if case['steps']:
        state['first'] = tokens[:, 0].contiguous()
        state['chosen'] = torch.zeros(case['steps'], case['rows'], dtype=torch.int32, device='cuda')
    return state


def run(state):
    m, p = state['m'], state['pos']
    m.seek(p)
    if state['steps']:
        m.x.copy_(state['first'])
        m.step(state['steps'], state['chosen'])
        chosen, n = state['chosen'], state['steps']
    else:
        m.prefill(state['tokens'])
        chosen, n = m.x, state['prompt']
    return dict(logits=m.logits(), tokens=chosen, keys=m.keys[:, :, p:p + n], vals=m.vals[:, :, p:p + n])


def work(case):
    cfg, rows, pos = SHAPES[case['model']], case['rows'], case['pos']
    d, layers = cfg.n_embd, cfg.n_layer
    layer_params = 4 * d * d + 2 * d * cfg.n_inner
    weights = 2 * (layers * (layer_params + 3 * d + d + cfg.n_inner + d + 4 * d) + cfg.vocab * d + 2 * d)
    row_bytes = 2 * 2 * layers * d                 # one position's keys and values
    if case['kind'] == 'decode':
        n = case['steps']
        contexts = sum(pos + k + 1 for k in range(n))
        nbytes = n * (weights + rows * (2 * d + row_bytes + 4)) + rows * (contexts - n) * row_bytes
        flops = n * 2 * rows * (layers * layer_params + cfg.vocab * d)
    else:
        n = case['prompt']
        contexts = sum(pos + k + 1 for k in range(n))
        nbytes = weights + rows * n * (4 + row_bytes) + rows * pos * row_bytes
        flops = 2 * rows * (n * layers * layer_params + cfg.vocab * d)
    return {'bytes': nbytes + 4 * rows * cfg.vocab, 'flops': flops + 4 * rows * contexts * layers * d}


def tolerance(case):
    # Measured against exact(): logits 3e-7 .. 5e-6 off for decode steps, 6e-6 .. 6e-5 for prefills (fp32
    # sums and 22-bit activations leave about 1e-6; the rest comes from new cache rows that lie next to an
    # fp16 rounding boundary and go the other way). The cache rows themselves are rounded to fp16 (2.1e-4
    # off); where two implementations differ there, it is by one place, 2^-10 of the value at most.
    return {'rel': 2.5e-4, 'max': 4e-3, 'differ': 0.01}


def _norm(z, w, b):
    c = z - z.mean(-1, keepdim=True)
    return c / torch.sqrt((c * c).mean(-1, keepdim=True) + 1e-5) * w.double() + b.double()


def _forward(sd, cfg, tokens, pos, cache):
    """One pass in 64 bits over tokens [rows, n] at positions pos ..; ``cache`` holds each layer's keys
    and values [rows, pos, heads, 64] and gets the new rows, which attention reads as the fp16 cache
    holds them. Returns the last position's logits and the new rows before that rounding."""
    rows, n = tokens.shape
    heads, width = cfg.n_head, cfg.head_dim
    wte = sd['transformer.wte.weight']
    z = wte[tokens.long()].double() + sd['transformer.wpe.weight'][pos:pos + n].double()
    made = []
    for i in range(cfg.n_layer):
        def product(a, name, i=i):
            p = f'transformer.h.{i}.{name}'
            return a @ sd[p + '.weight'].double() + sd[p + '.bias'].double()

        def norm(a, name, i=i):
            return _norm(a, sd[f'transformer.h.{i}.{name}.weight'], sd[f'transformer.h.{i}.{name}.bias'])

        q, *kv = (t.reshape(rows, n, heads, width) for t in product(norm(z, 'ln_1'), 'attn.c_attn').chunk(3, -1))
        made.append(kv)
        cache[i] = [torch.cat((old, new.half()), 1) for old, new in zip(cache[i], kv)]
        out = torch.empty_like(z)
        later = torch.ones(n, pos + n, dtype=torch.bool, device=z.device).triu(pos + 1)
        for b in range(rows):
            k, v = (c[b].double().transpose(0, 1).contiguous() for c in cache[i])
            s = (q[b].transpose(0, 1).contiguous() @ k.transpose(1, 2).contiguous()) / 8.0
            w = torch.softmax(s.masked_fill(later, -math.inf), -1)
            out[b] = (w @ v).transpose(0, 1).reshape(n, -1)
        z = z + product(out, 'attn.c_proj')
        u = product(norm(z, 'ln_2'), 'mlp.c_fc')
        g = 0.5 * u * (1.0 + torch.tanh(0.7978845608028654 * (u + 0.044715 * u ** 3)))
        z = z + product(g, 'mlp.c_proj')
    y = _norm(z[:, -1], sd['transformer.ln_f.weight'], sd['transformer.ln_f.bias'])
    return y @ wte.double().t(), made


def exact(case, seed):
    weights, tokens, past = _inputs(case, seed)
    cfg, sd = weights.config, weights.state_dict()
    cache = [[p[:, i] for p in past] for i in range(cfg.n_layer)]
    del past
    x, chosen, rows = tokens, [], []
    for k in range(max(1, case['steps'])):
        logits, made = _forward(sd, cfg, x, case['pos'] + k, cache)
        rows.append(made)
        x = logits.argmax(-1, keepdim=True).int()
        chosen.append(x[:, 0])
    keys, vals = (torch.stack([torch.cat([r[i][j] for r in rows], 1) for i in range(cfg.n_layer)], 1)
                  for j in range(2))
    return dict(logits=logits, tokens=torch.stack(chosen) if case['steps'] else chosen[0], keys=keys, vals=vals)
