"""Multi-token prefill: a prompt's positions go through each layer together.

The reference feeds a prompt one token per launch (reference
``bench/g0_bench.py:172-173``): P decode steps, each reading every weight.
Here the B rows' P positions form one M = B * P row batch and each layer is
a handful of ordinary launches (``hip/prefill.hip``): LayerNorm, the qkv
product writing the key/value cache rows, causal attention over the cache,
the out-projection with its residual, LayerNorm, the widening product with
GELU, the narrowing product with its residual. The products run on the
matrix cores. Only the last position of each row goes through the final
LayerNorm and the tied output head; its argmax becomes the next input.

Afterwards the model is in the state P decode steps would leave: cache rows
t0 .. t0 + P - 1 written, ``x`` the token chosen after the last prompt token,
``t`` advanced by P, ``logits()`` that step's logits.

The same launch sequence with one position per row is the layered decode
engine (``Prefill.decode``, replayed from a captured HIP graph). All products
read weights packed once in the matrix cores' operand order
(``frag_weights``) and activations that the LayerNorms, attention and the
widening product's GELU write in that order: up to 64 rows ``pf_mgemm*``,
whose waves split the fold, beyond ``pf_pgemm*`` in output tiles.
"""
from __future__ import annotations

import ctypes
import math
from pathlib import Path

from .launch import compile_code, lib, ok, track, unload

PREFILL_SRC = Path(__file__).resolve().parent / 'hip' / 'prefill.hip'
PRELUDE_SRC = Path(__file__).resolve().parent / 'hip' / 'prelude.h'
BLOCK = 256
CHUNK = 64                    # products' fold lengths are multiples of this (two 32-deep k-steps)
HEAD = 64
KERNELS = ('pf_embed_ln', 'pf_ln', 'pf_lnm8', 'pf_lnm16', 'pf_mgemm1', 'pf_mgemm2', 'pf_mgemm4', 'pf_mgemm1n',
           'pf_mgemm2n', 'pf_mgemm4n', 'pf_pgemm128', 'pf_pgemm64', 'pf_pgemm64w', 'pf_pgemm32', 'pf_pgemm32o',
           'pf_reduce', 'pf_reduce_ln', 'pf_reduce_frag', 'pf_attn', 'pf_attn16', 'pf_attn1', 'pf_attn1s', 'pf_mhead1',
           'pf_mhead2', 'pf_mhead4', 'pf_argmax_part', 'pf_argmax')
ARGMAX_SPLIT = 32             # blocks per row of the output-head argmax (same box, 16 -> 32: GPT-2 small 32 rows
                              # 547.6 -> 545.8 us per step, 8 rows 396.3 -> 395.5, XL 64 rows even)
# output tiles of the products beyond FEW_ROWS rows: 16-row tiles, 16-column tiles and waves of a block
PG_TILES = {'pf_pgemm128': (8, 16, 8), 'pf_pgemm64': (4, 8, 8), 'pf_pgemm64w': (4, 8, 4), 'pf_pgemm32': (2, 4, 4)}
MODE_PLAIN, MODE_RESID, MODE_GELU, MODE_QKV = 0, 1, 2, 3
FEW_ROWS = 64                 # products of up to this many rows are pf_mgemm*, of more pf_pgemm*
MG_WAVES = 8                  # waves of a pf_mgemm block ...
MG_TILES = {1: 1, 2: 1, 4: 2}  # ... and the 16-column tiles it makes, by 16-row tiles (pf_mgemm1/2/4's MN)
MG_BLOCKS = 200               # such a product splits its fold so that it has about this many blocks, ...
MG_MIN_STEPS = 16             # ... each part at least this many 32-deep k-steps (two per wave)
MG_MIN_STEPS_LN = 8           # ... or this many for a residual product whose reduction makes the next LayerNorm
                              # (its split adds no launch; same box, 16 / 12 / 8: XL B=64 3.089 / 3.057 / 3.059
                              # ms per step, small B=32 with 1024 positions 0.620 / 0.610 / 0.608)
MEM_CACHE_BYTES = 256 << 20   # the device's memory-side cache: decode products of a model whose weights are
                              # larger load them nontemporal (same box: XL B=64 3.000 -> 2.944 ms per step,
                              # medium B=16 0.958 -> 0.916; GPT-2 small's 247 MB stay in that cache between
                              # steps, nontemporal there: 32 rows 0.548 -> 0.553)
LNM_ROWS = 1536               # LayerNorms of at least this many rows take a block per 16 rows (pf_lnm*; us a
                              # launch, block per row / per 16 rows: 999 x 768 6.3 / 7.3, 2048 x 768 8.7 / 7.7, 999 x
                              # 1600 8.3 / 12.7, 2048 x 1600 13.0 / 13.7, 4096 x 1600 24.0 / 15.9)
ORDERED_TOKENS, ORDERED_LAYERS = 8, 24      # see ordered()
ATTN_SPLIT_BLOCKS = 512       # prefill attention with at most this many blocks of 16 queries (two per CU, all
                              # resident) splits each one's positions over its waves (pf_attn16). us a launch, pf_attn
                              # / pf_attn16, GPT-2 small: 1 x 200 after 700 positions (156 such blocks) 25.3 / 10.9,
                              # 20 x 32 after 365 (480) 14.6 / 11.9, 60 x 3 (720) 6.6 / 6.8, 8 x 128 (768) 7.5 / 10.9
ATTN_ONE_PASS_BLOCKS = 1024   # decode passes with at most this many (row, head) blocks read each cache row in
                              # one pass (pf_attn1s), more in two (pf_attn1: keys, then values; fewer
                              # registers, more blocks resident). Same box, two -> one pass: small 16 / 24 rows
                              # (192 / 288 blocks, 448 positions) 0.450 -> 0.436 / 0.479 -> 0.466 ms per step,
                              # 32 rows (384, 1024 positions) 0.666 -> 0.637; XL 64 rows (1600) 3.110 -> 3.128


def supported(D, H, F):
    """Shapes the prefill kernels take: 64-wide heads and products whose fold
    lengths are multiples of the 64-deep chunk a product stages at a time."""
    return H * HEAD == D and D % CHUNK == 0 and F % CHUNK == 0 and D <= 8 * BLOCK


def _mtiles(rows: int) -> int:
    """16-row tiles of the fragment-order activations of ``rows`` rows: up to
    64 rows those of the kernels for few rows (pf_mgemm1 / 2 / 4)."""
    t = -(-rows // 16)
    return t if t > 4 else 1 if t <= 1 else 2 if t == 2 else 4


def pgemm_us(name, M, N, K, ks):
    """Estimated time of a product of more than FEW_ROWS rows, in us: a fixed
    part, and for each 32-deep k-step of a block a time by how many blocks a
    CU gets (r). Fitted to the products of the three models at 65 to 24576
    rows, timed alone and inside whole prefills (where weights and activations
    come from farther away): the choice by it is within 2% of the fastest on
    average, some 20-30% off at a few row counts (small at 1024 rows, the
    out-projection: 9.2 against 7.5 us); e.g. (measured alone,
    us) qkv of GPT-2 small at 128 rows 6.6 / 11.1 / 22.6 in 32 x 64 / 64 x 128 /
    128 x 256 tiles, at 1024 rows 17.8 / 18.5 (four waves: 17.4) / 24.1, at
    24576 rows 280 / 207 (177) / 174; narrowing of XL at 8192 rows 552 / 405
    (373) / 332."""
    bm, bn, _ = PG_TILES[name]
    b = -(-M // (16 * bm)) * -(-N // (16 * bn)) * ks / 256
    k = K / 32 / ks
    r = math.ceil(b) if b <= 6 else b
    if name == 'pf_pgemm128':                           # one block per CU at a time
        us = math.ceil(b) * (8.61 + 0.719 * k)
    elif name == 'pf_pgemm64':
        us = 2.25 + k * max(0.448, 0.295 * r) + 1.14 * b
    elif name == 'pf_pgemm64w':                         # (reads its weights through L2, dearer where they are deep)
        us = 2.39 + k * max(0.662, 0.309 * r * (1 + 8.7e-6 * K) - 0.021)
    else:
        us = 3.43 + k * max(0.162, 0.11 * r * (1 + 8.9e-6 * K))
    # the parts of a split fold are stored and read back (by the launch that makes the LayerNorm either way)
    return us + ((1.43 * ks - 0.665) * M * N * 1e-6 - 0.25 if ks > 1 else 0)


def pgemm_plan(M, N, K, split):
    """Kernel and fold parts of a product of more than FEW_ROWS rows
    (``split``: whether its fold may be split): the least ``pgemm_us``."""
    return min(((name, ks) for name in PG_TILES for ks in ((1, 2, 3, 4, 6) if split else (1,)) if K // 64 >= 2 * ks
                or ks == 1), key=lambda c: pgemm_us(c[0], M, N, K, c[1]))


def ordered(P, L, t0):
    """Whether a prompt of P tokens at position t0 in a model of L layers keeps
    the order of sums that prompts had in products of 64 x 64 tiles with split
    folds and in an attention of one wave a query (``ordered_parts``,
    ``pf_pgemm32o``, ``pf_attn_short``), so that its results stay the same bit
    for bit. From an empty cache a short prompt's attention averages over few
    positions, so a new cache row that lies next to an fp16 rounding boundary
    and goes the other way is carried on almost undiminished, layer after
    layer: with any other order of sums XL's cache rows come out 2.2e-4 ..
    2.9e-4 apart (2-norm) at 2-6 tokens, about the 2.5e-4 by which
    perf/cases.py lets results differ; 2.1e-4 at 8, 1.6e-4 at 16; after one
    position 1.4e-4 .. 1.8e-4, after eight 0.8e-4; medium's 1.5e-4 .. 2.1e-4 at
    2-8, GPT-2 small's below 1.5e-4. It is a matter of sameness alone: these
    sums are no nearer to 64 bits (cache rows, XL 3 x 3 2.47e-4 against 2.44e-4,
    3 x 7 2.19e-4 against 2.09e-4) and take longer (XL 4 x 3 2.54 ms against
    2.07)."""
    return t0 == 0 and 1 < P <= ORDERED_TOKENS and L >= ORDERED_LAYERS


def ordered_parts(M, N, K):
    """Fold parts of an ordered product: about 384 output tiles of 64 x 64
    times parts, each part at least 256 deep. (So the order is that of the
    whole batch's size: the same for all batches of up to 64 rows in all.)"""
    return max(1, min(-(-384 // (-(-M // 64) * -(-N // 64))), K // 256))


def prefill_attn(B, P, H, ordered=False):
    """Kernel and blocks of the prefill attention of B rows of P positions."""
    few = B * H * -(-P // 16)
    return ('pf_attn16', few) if ordered or few <= ATTN_SPLIT_BLOCKS else ('pf_attn', B * H * -(-P // 64))


def frag_weights(Wt):
    """Weights [.., N, K] (row n: output n's K weights) in the decode
    products' fragment order [.., N/16, K/32, 64, 8]: element (n, k) at
    n-tile n // 16, k-step k // 32, lane 16 * ((k % 32) // 8) + n % 16,
    position k % 8 (the B operand of v_mfma_f32_16x16x32_f16 as a lane
    holds it). N is padded with zero rows to a multiple of 16."""
    import torch
    *lead, N, K = Wt.shape
    Np = -(-N // 16) * 16
    if Np != N:
        Wt = torch.cat([Wt, Wt.new_zeros(*lead, Np - N, K)], dim=-2)
    f = Wt.reshape(*lead, Np // 16, 16, K // 32, 4, 8)
    n = len(lead)
    return f.permute(*range(n), n, n + 2, n + 3, n + 1, n + 4).reshape(*lead, Np // 16, K // 32, 64, 8)


def frag_offset(M16: int, K: int, plane: int, m: int, k: int) -> int:
    """Half index of activation element (m, k) in fragment order (the
    layout pf_frag_put8 writes: plane, m-tile, k-step, lane, 8; M16 rows in
    16-row tiles)."""
    MT, KT = M16 // 16, K // 32
    return (((plane * MT + m // 16) * KT + k // 32) * 64 + ((k % 32) // 8) * 16 + m % 16) * 8 + k % 8


def prefill_source(tmax: int) -> str:
    return (f'#define VBLOCK {BLOCK}\n#define PF_TMAX {tmax}\n' + PRELUDE_SRC.read_text() + '\n'
            + PREFILL_SRC.read_text())


class _Args:
    """A kernel argument array for the C-ABI launch: pointers to each value."""

    def __init__(self, vals):
        self.vals = vals
        ptrs = [ctypes.cast(ctypes.pointer(v), ctypes.c_void_p) for v in vals]
        self.array = (ctypes.c_void_p * len(ptrs))(*ptrs)


def _p(t):
    """A pointer argument: a tensor's, or one given as it is."""
    if isinstance(t, ctypes.c_void_p):
        return t
    return ctypes.c_void_p(t.data_ptr() if t is not None else 0)


def _i(v):
    return ctypes.c_int(int(v))


class Prefill:
    """The prefill kernels bound to one ``VestaGPT2``'s weights and cache."""

    def __init__(self, model, graphs=True):
        self.m = model
        self.graphs = graphs           # layered decode steps replay a captured HIP graph
        if not supported(model.D, model.H, model.W['fcw'].shape[2]):
            raise ValueError(f'prefill kernels need 64-wide heads and widths that are multiples of 64 '
                             f'(d={model.D}, H={model.H})')
        self.code = compile_code(prefill_source(model.tmax))
        L = lib()
        mod = ctypes.c_void_p()
        ok(L.vh_module_load(self.code, ctypes.byref(mod)), 'prefill module load')
        self.mod = mod
        track(self)
        self.fn = {}
        for name in KERNELS:
            fn = ctypes.c_void_p()
            ok(L.vh_module_get_function(mod, name.encode(), ctypes.byref(fn)), name)
            self.fn[name] = fn
        import torch
        self.err = torch.zeros(1, dtype=torch.int32, device='cuda')   # raised by a product that met an
                                                                     # activation beyond the fp16 range
        self._bufs = {}
        self._own = {}
        self._ws = None
        self._ws_at = ctypes.c_void_p()
        self._graph = None
        self._plans = {}
        self._plan = []

    def check(self):
        """Raise if a product of an earlier launch met an activation beyond the
        fp16 range its matrix-core path can carry (one synchronisation); the
        word is cleared first."""
        if int(self.err.item()):
            self.err.zero_()
            raise RuntimeError('layered engine: an activation beyond the fp16 range (65504) reached a matrix-core '
                               'product; the results are invalid')

    def close(self):
        if getattr(self, 'mod', None) is not None and self.mod.value:
            try:
                self._graph = None          # a captured graph holds launches of this module
                unload(self.mod)
            except Exception:
                pass
            self.mod = None

    def __del__(self):
        self.close()

    def _launch(self, name, grid, vals, block=BLOCK):
        """Record one launch of the plan being built."""
        self._plan.append((name, self.fn[name], int(grid), _Args(vals), int(block)))

    def _buffers(self, M):
        """Activation buffers for M rows (one set per row count, kept): the
        residual Z, the queries Q, and the fragment-order activations AF of
        the products over d (LayerNorm and attention outputs) and GF of the
        one over the feed-forward width (GELU outputs). These are zeroed
        once: rows past M are never written."""
        import torch
        if M not in self._bufs:
            m = self.m
            F = m.W['fcw'].shape[2]
            rows = 16 * _mtiles(M)
            f32 = dict(dtype=torch.float32, device='cuda')
            h16 = dict(dtype=torch.float16, device='cuda')
            self._bufs[M] = dict(Z=torch.empty(M, m.D, **f32), Q=torch.empty(M, m.D, **f32),
                                 AF=torch.zeros(2 * rows * m.D, **h16), GF=torch.zeros(2 * rows * F, **h16),
                                 CF=torch.zeros(2 * 16 * _mtiles(m.B) * m.D, **h16),
                                 tok=torch.empty(M, dtype=torch.int32, device='cuda'),
                                 apv=torch.empty(m.B * ARGMAX_SPLIT, **f32),
                                 api=torch.empty(m.B * ARGMAX_SPLIT, dtype=torch.int32, device='cuda'))
        return self._bufs[M]

    def _frag(self, name):
        """Weight ``name`` in the products' fragment order
        ([L,] n-tile, k-step, lane, 8; see hip/prefill.hip), made on first use
        and held. Layer weights are stored [L, in, out]; the output head
        ``wte`` [V, d] is already [out, in] and gets zero rows up to a
        multiple of 16."""
        key = name + '__f'
        if key not in self._own:
            W = self.m.W[name]
            self._own[key] = frag_weights(W) if name == 'wte' else frag_weights(W.transpose(1, 2))
        return self._own[key]

    def _mgemm(self, Af, K, wname, layer, N, mode, bias=None, out=None, ldo=0, F=None, ln=None, M=1, P=1):
        """One product of at most 64 rows (``pf_mgemm*``) over M rows (P
        positions each of M / P rows): A in fragment order (Af), weights
        ``wname`` (layer ``layer``) in fragment order. With a split fold the parts are added by a second launch: ``pf_reduce_ln``
        for a residual product followed by the LayerNorm ``ln`` = (w, b, F_out)
        (returns True: that LayerNorm is done), ``pf_reduce_frag`` for the
        GELU product, ``pf_reduce`` otherwise."""
        m = self.m
        KT, NT = K // 32, -(-N // 16)
        mt = _mtiles(M)
        if K % 32 or M > 16 * mt or mt > 4:
            raise ValueError(f'product {wname}: K={K} must be a multiple of 32 and M={M} at most 64')
        nb = -(-NT // MG_TILES[mt])
        steps = MG_MIN_STEPS_LN if mode == MODE_RESID and ln is not None else MG_MIN_STEPS
        ks = max(1, min(round(MG_BLOCKS / nb), KT // steps))
        ws = self._workspace(ks * M * N) if ks > 1 else None
        Wf = self._frag(wname)
        Wf = Wf[layer] if layer is not None else Wf
        # the extents pf_mgemm* indexes, checked before the launch is recorded
        if Af.numel() < 2 * 16 * mt * K or Wf.numel() < NT * KT * 512:
            raise ValueError(f'product {wname}: operands smaller than {M}x{K} activations / {N}x{K} weights')
        if mode == MODE_GELU and (N % 32 or F is None or F.numel() < 2 * 16 * mt * N):
            raise ValueError(f'product {wname}: GELU output needs a fragment buffer of {M}x{N}, N % 32 == 0')
        if mode == MODE_PLAIN:
            raise ValueError(f'product {wname}: the output head of up to 64 rows is pf_mhead*')
        if mode == MODE_RESID and ln is not None and ldo != N:
            raise ValueError(f'product {wname}: a LayerNorm over rows of {N} needs their pitch to be {N}')
        if mode != MODE_GELU and out.numel() < M * ldo:
            raise ValueError(f'product {wname}: output smaller than {M} rows of {ldo}')
        t_args = [_p(m.keys), _p(m.vals), _i(P), _p(m.t), _i(layer or 0), _i(m.L), _i(m.tmax)]
        self._launch(f'pf_mgemm{mt}' + ('n' if self._weights_nt() else ''), nb * ks,
                     [_p(Af), _p(Wf), _i(KT), _i(NT), _i(ks), _p(bias), _i(M), _i(N), _i(mode), _p(out), _i(ldo)]
                     + t_args + [_p(ws), _p(F), _p(self.err)], block=MG_WAVES * 64)
        return self._reduce(ws, ks, bias, M, N, mt, mode, out, ldo, P, layer, F, ln)

    def _pgemm(self, Af, K, wname, layer, N, mode, bias=None, out=None, ldo=0, F=None, ln=None, M=1, P=1, ks=None):
        """One product of any number of rows (``pf_pgemm*``), as ``_mgemm``.
        With ``ks`` None only a residual product with a LayerNorm after it
        splits its fold (its reduction adds no launch); else it is made in
        ``ks`` parts, each part's sum whole (``pf_pgemm32o``)."""
        m = self.m
        KT, NT, MT = K // 32, -(-N // 16), _mtiles(M)
        if ks is None:
            name, ks = pgemm_plan(M, N, K, mode == MODE_RESID and ln is not None)
            bm, bn, waves = PG_TILES[name]
        else:
            name, (bm, bn, waves) = 'pf_pgemm32o', PG_TILES['pf_pgemm32']
        ws = self._workspace(ks * M * N) if ks > 1 else None
        Wf = self._frag(wname)
        Wf = Wf[layer] if layer is not None else Wf
        # the extents pf_pgemm* indexes, checked before the launch is recorded
        if K % 64 or MT * 16 < M:
            raise ValueError(f'product {wname}: K={K} must be a multiple of 64')
        if Af.numel() < 2 * 16 * MT * K or Wf.numel() < NT * KT * 512:
            raise ValueError(f'product {wname}: operands smaller than {M}x{K} activations / {N}x{K} weights')
        if mode == MODE_GELU and (N % 32 or F is None or F.numel() < 2 * 16 * MT * N):
            raise ValueError(f'product {wname}: GELU output needs a fragment buffer of {M}x{N}, N % 32 == 0')
        if mode != MODE_GELU and out.numel() < (M - 1) * ldo + (N // 3 if mode == MODE_QKV else N):
            raise ValueError(f'product {wname}: output smaller than {M} rows of {ldo}')
        if mode == MODE_PLAIN and ks > 1:
            raise ValueError(f'product {wname}: a plain product is made whole')
        if mode == MODE_RESID and ln is not None and ldo != N:
            raise ValueError(f'product {wname}: a LayerNorm over rows of {N} needs their pitch to be {N}')
        if mode != MODE_PLAIN and (N % 64 or ldo % 4 or bias is None):
            raise ValueError(f'product {wname}: N={N} must be a multiple of 64, the output pitch of 4, with a bias')
        tiles = -(-MT // bm) * -(-NT // bn) * ks
        self._launch(name, 8 * -(-tiles // 8),
                     [_p(Af), _p(Wf), _i(MT), _i(KT), _i(NT), _i(ks), _p(bias), _i(M), _i(N), _i(mode), _p(out),
                      _i(ldo), _p(m.keys), _p(m.vals), _i(P), _p(m.t), _i(layer or 0), _i(m.L), _i(m.tmax), _p(ws),
                      _p(F), _p(self.err)], block=waves * 64)
        return self._reduce(ws, ks, bias, M, N, MT, mode, out, ldo, P, layer, F, ln)

    def _reduce(self, ws, ks, bias, M, N, MT, mode, out, ldo, P, layer, F, ln):
        """The launch that adds a split product's parts, if there are any;
        returns whether it made the LayerNorm ``ln`` too."""
        m = self.m
        if ks == 1:
            return False
        if mode == MODE_RESID and ln is not None:
            w, b, Fo = ln
            self._launch('pf_reduce_ln', M, [_p(ws), _i(ks), _p(bias), _i(M), _i(N), _p(out), _p(w), _p(b), _p(Fo),
                                             _i(MT), _p(self.err)])
            return True
        if mode == MODE_GELU:
            self._launch('pf_reduce_frag', -(-M * (N // 8) // BLOCK), [_p(ws), _i(ks), _p(bias), _i(M), _i(N), _p(F),
                                                                       _i(MT), _p(self.err)])
        else:
            self._launch('pf_reduce', -(-M * N // BLOCK), [_p(ws), _i(ks), _p(bias), _i(M), _i(N), _i(mode), _p(out),
                                                            _i(ldo), _p(m.keys), _p(m.vals), _i(P), _p(m.t),
                                                            _i(layer or 0), _i(m.L), _i(m.tmax)])
        return False

    def _product(self, Af, K, wname, layer, N, mode, M, ordered=False, **kw):
        """A product on the kernels for its row count (True: the LayerNorm
        that follows it is done)."""
        a = (Af, K, wname, layer, N, mode)
        if ordered:
            return self._pgemm(*a, M=M, ks=ordered_parts(M, N, K), **kw)
        return (self._mgemm if M <= FEW_ROWS else self._pgemm)(*a, M=M, **kw)

    def _weights_nt(self):
        """Whether the decode products load their weights nontemporal
        (``pf_mgemm*n``): when the model's weights do not fit the memory-side
        cache."""
        return getattr(self.m, 'weight_bytes', 0) > MEM_CACHE_BYTES

    def _mhead(self, Af, K, N, out, M):
        """The output head over M rows (``pf_mhead*``): logits [M, N] = A wte^T,
        A in fragment order (Af), the packed head weights; a block of
        MG_WAVES waves per 2 MG_WAVES column tiles, each wave over the whole
        fold."""
        KT, NT = K // 32, -(-N // 16)
        Wf = self._frag('wte')
        mt = _mtiles(M)
        if K % 32 or M > 16 * mt or mt > 4 or Af.numel() < 2 * 16 * mt * K or Wf.numel() < NT * KT * 512 \
                or out.numel() < M * N:
            raise ValueError(f'output head: operands do not cover {M}x{K} activations, {N}x{K} weights')
        self._launch(f'pf_mhead{mt}', -(-NT // (2 * MG_WAVES)),
                     [_p(Af), _p(Wf), _i(KT), _i(NT), _i(M), _i(N), _p(out), _i(N)], block=MG_WAVES * 64)

    def _attn1(self):
        """The decode attention kernel for this model's rows and heads."""
        return 'pf_attn1s' if self.m.B * self.m.H <= ATTN_ONE_PASS_BLOCKS else 'pf_attn1'

    def _workspace(self, n):
        """Partial tiles of split products: one buffer, grown to the largest
        need (launches on one stream run one after another). Returns the
        argument that all launches share, which follows the buffer when it
        grows."""
        import torch
        if self._ws is None or self._ws.numel() < n:
            self._graph = None          # a captured graph holds the old pointer
            self._ws = torch.empty(n, dtype=torch.float32, device=self.err.device)
            self._ws_at.value = self._ws.data_ptr()
        return self._ws_at

    def _plan_for(self, key, buf, B, P, tok, fixed=False):
        """The launch plan ``key``, built on first use."""
        if key not in self._plans:
            self._plan = []
            self._build(buf, B, P, tok, fixed)
            self._plans[key] = self._plan
        return self._plans[key]

    def _replay(self, plan):
        import torch
        stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        L = lib()
        for name, fn, grid, a, block in plan:
            ok(L.vh_launch(fn, grid, block, 0, stream, a.array), name)

    def run(self, prompt, t0=0):
        """Prefill ``prompt`` (int32 device tensor [B, P]) at positions t .. t + P - 1
        (t the model's position counter, read and advanced on the device;
        ``t0``: the host's copy of it, for the choice of kernels alone).

        The launch sequence with its argument arrays is built once per P and
        order of sums (``ordered``) and replayed: every pointer it holds
        (weights, cache, this object's activation buffers and prompt copy)
        stays fixed."""
        B, P = prompt.shape
        buf = self._buffers(B * P)
        buf['tok'].copy_(prompt.reshape(-1))
        fixed = ordered(P, self.m.L, t0)
        self._replay(self._plan_for((P, fixed), buf, B, P, buf['tok'], fixed))

    def decode(self, n, tokens=None):
        """``n`` greedy decode steps, each one pass with P = 1 over the
        model's input ``x`` (the last pass's argmax): the layer-at-a-time
        path for shapes the persistent kernel does not fit. ``tokens`` (a
        contiguous int32 device tensor of at least n * B ids, any shape, e.g.
        [n, B]) receives each step's chosen tokens, step k at flat offsets
        k * B .. k * B + B - 1."""
        m = self.m
        flat = None
        if tokens is not None:
            if not (tokens.is_cuda and tokens.dtype == m.x.dtype and tokens.is_contiguous()):
                raise TypeError('tokens must be a contiguous int32 device tensor')
            if tokens.numel() < n * m.B:
                raise ValueError(f'tokens holds {tokens.numel()} ids, {n * m.B} needed')
            flat = tokens.view(-1)
        buf = self._buffers(m.B)
        plan = self._plan_for('decode', buf, m.B, 1, m.x)
        step = lambda: self._replay(plan)       # noqa: E731
        if self.graphs:
            if self._graph is None or self._graph[0] is not plan:
                self._graph = (plan, self._capture(plan))
            step = self._graph[1].replay
        for k in range(n):
            step()
            if flat is not None:
                flat[k * m.B:(k + 1) * m.B].copy_(m.x)

    def _capture(self, plan):
        """One decode pass recorded as a HIP graph: a step is then one graph
        launch instead of some hundred kernel launches from the host. The pass
        has no memory sets or host reads, and every pointer it holds stays
        fixed (the position is read on the device)."""
        import torch
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            self._replay(plan)
        return g

    def _build(self, buf, B, P, tok, fixed):
        """The launches of one pass: B rows of P positions each (P = 1: a
        decode step; ``fixed``: the order of sums is kept, see ``ordered``).
        LayerNorm and attention write their outputs as the next product's
        fragment-order activations (AF), the widening product its GELU outputs
        as the narrowing one's (GF)."""
        m = self.m
        M, D, H, L = B * P, m.D, m.H, m.L
        F = m.W['fcw'].shape[2]
        V = m.W['wte'].shape[0]
        W = m.W
        Z, Q, AF, GF, err = buf['Z'], buf['Q'], buf['AF'], buf['GF'], self.err
        mt = _mtiles(M)

        def norm(w, b, to, rows, row0=0, stride=1):
            if rows >= LNM_ROWS and stride == 1:
                self._launch('pf_lnm8' if D <= 1024 else 'pf_lnm16', -(-rows // 16),
                             [_p(Z), _i(rows), _i(D), _p(w), _p(b), _p(to), _i(_mtiles(rows)), _p(err)])
                return
            self._launch('pf_ln', rows, [_p(Z), _i(row0), _i(stride), _p(w), _p(b), _i(D), _p(to), _i(_mtiles(rows)),
                                         _p(err)])
        self._launch('pf_embed_ln', M, [_p(tok), _i(P), _p(m.t), _p(W['wte']), _p(W['wpe']), _p(Z), _i(D), _i(V),
                                        _i(W['wpe'].shape[0]), _p(W['ln1w'][0]), _p(W['ln1b'][0]), _p(AF), _i(mt),
                                        _p(err)])
        for layer in range(L):
            def lw(name, layer=layer):
                return W[name][layer]
            self._product(AF, D, 'qkvw', layer, 3 * D, MODE_QKV, bias=lw('qkvb'), out=Q, ldo=D, M=M, P=P,
                          ordered=fixed)
            cache = [_p(Q), _p(m.keys), _p(m.vals)]
            if P == 1:          # a block per (row, head) (GPT-2 small, 32 rows, 1024 positions:
                                # 1.32 -> 1.07 ms per step against a wave per (row, head))
                self._launch(self._attn1(), B * H, cache + [_p(m.t), _i(layer), _i(L), _i(m.tmax), _i(H), _p(AF),
                                                            _i(mt), _p(err)])
            else:
                name, blocks = prefill_attn(B, P, H, fixed)
                self._launch(name, 8 * -(-blocks // 8), cache + [_i(B), _i(P), _p(m.t), _i(layer), _i(L), _i(m.tmax),
                                                                 _i(H), _p(AF), _i(mt), _p(err)])
            if not self._product(AF, D, 'ow', layer, D, MODE_RESID, bias=lw('ob'), out=Z, ldo=D,
                                 ln=(lw('ln2w'), lw('ln2b'), AF), M=M, ordered=fixed):
                norm(lw('ln2w'), lw('ln2b'), AF, M)
            self._product(AF, D, 'fcw', layer, F, MODE_GELU, bias=lw('fcb'), F=GF, M=M, ordered=fixed)
            last = layer + 1 == L
            nxt = (W['lnfw'], W['lnfb'], AF) if last else (lw('ln1w', layer + 1), lw('ln1b', layer + 1), AF)
            normed = self._product(GF, F, 'pw', layer, D, MODE_RESID, bias=lw('pb'), out=Z, ldo=D,
                                   ln=nxt if P == 1 or not last else None, M=M, ordered=fixed)
            if not normed and not (last and P > 1):
                norm(*nxt, M)
        if P > 1:               # the final norm: each row's last position
            norm(W['lnfw'], W['lnfb'], buf['CF'], B, P - 1, P)
        logit, nxt = m.logits(), m.next()
        head = buf['CF'] if P > 1 else AF
        if B <= FEW_ROWS:
            self._mhead(head, D, V, logit, B)
        else:
            self._pgemm(head, D, 'wte', None, V, MODE_PLAIN, out=logit, ldo=V, M=B)
        self._launch('pf_argmax_part', B * ARGMAX_SPLIT, [_p(logit), _i(V), _i(ARGMAX_SPLIT), _p(buf['apv']),
                                                           _p(buf['api'])])
        self._launch('pf_argmax', B, [_p(buf['apv']), _p(buf['api']), _i(ARGMAX_SPLIT), _p(m.x), _p(nxt), _p(m.t),
                                      _i(P)])
