"""Workloads that stand for the framework's use, each through its public entry points, with float64 references.

Five kinds of case, by the key ``kind``:

* ``step``: the attention of one serving step over paged latent caches (``s6_layer.StepContext``, ``latent_query``,
  ``attend``): ``requests`` requests with histories of ``ctx_min``..``ctx_max`` tokens and ``chunk_min``..``chunk_max``
  new tokens each, ``layers`` layers with caches of their own, all four loops loop-major as the model runs them.
* ``writer``: the row writer and commit of a step (``s6_layer.write_commit``, all four loops of every layer).
* ``rows``: the rolling engine's single-query history over contiguous rows with a key mask
  (``history_gemm.history_attention``), forward.
* ``khop``: multi-query history attention of a K-hop replay, forward and backward
  (``history_gemm.causal_history_gemm``), in bf16 or in the default fp32 precision.
* ``mixed``: the rolling engine's joint attention of a chunk over its history blocks, forward and backward
  (``batched_engine.mixed_attention``), with the gradients of the chunk, of the packed rows and of the readers.

The serving kinds (``step``, ``writer``, ``rows``) run as a HIP graph that ``prepare`` captures, as serving engines
replay their steps; the training kinds run eagerly through autograd.
"""
from __future__ import annotations

import importlib
import math
import random
import types

import torch

PKG = 'hybrid-latent-attention_amd'
HEADS, HEAD_DIM, RANK, RANK1, WINDOW, BLOCK, LOOPS, HIDDEN = 16, 128, 512, 256, 32, 16, 4, 2048
MAX_POSITION = 65536
SCALE = HEAD_DIM ** -0.5
BF = torch.bfloat16
# the adapter's constants: the largest captured batch bounds the split steps, the token budget sizes the workspace
SPLIT_MAX_TOKENS, MAX_BATCHED_TOKENS = 512, 8192


def listed():
    step = dict(kind='step', chunk_min=1, chunk_max=1)
    return [
        # one interactive user: a decode step at a short context, bound by latency and launches
        dict(step, name='decode_b1_ctx1024', requests=1, ctx_min=1024, ctx_max=1024, layers=4),
        # ordinary serving: requests of many lengths share a decode step
        dict(step, name='decode_b32_ragged', requests=32, ctx_min=1024, ctx_max=8192, layers=2),
        # a full batch at 8K context: throughput serving, the benchmark's headline shape
        dict(step, name='decode_b64_ctx8192', requests=64, ctx_min=8192, ctx_max=8192, layers=2),
        # few users with long documents
        dict(step, name='decode_b8_ctx32768', requests=8, ctx_min=32768, ctx_max=32768, layers=2),
        # a K-hop step: a few new tokens per request on a long history
        dict(step, name='chunk3_b4_ctx8192', requests=4, ctx_min=8224, ctx_max=8224, chunk_min=3, chunk_max=3,
             layers=4),
        # chunked prefill of long prompts
        dict(step, name='prefill_b4_q512', requests=4, ctx_min=8224, ctx_max=8224, chunk_min=512, chunk_max=512,
             layers=1),
        # the writer of a full decode batch, and of a prefill step of 2048 tokens
        dict(kind='writer', name='writer_decode_b64', requests=64, chunk=1, layers=8),
        dict(kind='writer', name='writer_prefill_t2048', requests=4, chunk=512, layers=4),
        # the rolling engine's decode call: 8 rows of padded histories
        dict(kind='rows', name='rows_b8_n8192', batch=8, rows=8192, width=512),
        # K-hop replay training at the operator benchmark's length; bf16, and the default precision at an odd length
        dict(kind='khop', name='khop_bf16_w512', batch=4, length=2880, width=512, precision='bf16'),
        dict(kind='khop', name='khop_fp32_w256', batch=4, length=2045, width=256, precision='fp32'),
        # the rolling engine's training step on a chunk with a long and a short history block
        dict(kind='mixed', name='mixed_b8_n256', batch=8, chunk=256, block0=2048, block1=256, loop=2),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    """One more case of the same kinds: sizes over the whole range, odd ones among them."""
    kind = rng.choices(('step', 'writer', 'rows', 'khop', 'mixed'), (8, 2, 2, 2, 2))[0]
    while True:
        if kind == 'step':
            lo, hi = sorted((_log_int(rng, 40, 32768), _log_int(rng, 40, 32768)))
            q = rng.choices((1, _log_int(rng, 2, 15), _log_int(rng, 16, 512)), (4, 2, 3))[0]
            case = dict(kind=kind, requests=_log_int(rng, 1, 64), ctx_min=lo, ctx_max=hi,
                        chunk_min=rng.choice((1, q)), chunk_max=q, layers=rng.choice((1, 2)))
            tokens, rows = case['requests'] * q, case['requests'] * hi
            if tokens > 2048 or rows > 64 * 8192 or (q > 1 and tokens * hi > 2048 * 8192):
                continue
        elif kind == 'writer':
            case = dict(kind=kind, requests=_log_int(rng, 1, 64), chunk=rng.choice((1, _log_int(rng, 2, 512))),
                        layers=rng.choice((1, 2, 4)))
            if case['requests'] * case['chunk'] > 2048:
                continue
        elif kind == 'rows':
            case = dict(kind=kind, batch=_log_int(rng, 1, 16), rows=_log_int(rng, 300, 16384),
                        width=rng.choice((256, 512)))
            if case['batch'] * case['rows'] > 16 * 8192:
                continue
        elif kind == 'khop':
            case = dict(kind=kind, batch=_log_int(rng, 1, 6), length=_log_int(rng, 150, 2880),
                        width=rng.choice((256, 512)), precision=rng.choice(('bf16', 'bf16', 'fp32')))
            limit = 0.69e12 if case['precision'] == 'fp32' else 1.3e12
            if work(case)['flops'] > limit:
                continue
        else:
            case = dict(kind=kind, batch=_log_int(rng, 1, 8), chunk=_log_int(rng, 20, 256),
                        block0=_log_int(rng, 100, 2048), block1=_log_int(rng, 20, 256), loop=rng.randrange(LOOPS))
        return case


# ---- shapes ----------------------------------------------------------------------------------------------------

def _lengths(case):
    """Per request: history tokens and new tokens, the same for every seed (a case's work is fixed)."""
    rng = random.Random(f"{case['requests']} {case['ctx_min']} {case['ctx_max']} {case['chunk_min']} "
                        f"{case['chunk_max']}")
    hist = [rng.randint(case['ctx_min'], case['ctx_max']) for _ in range(case['requests'])]
    new = [rng.randint(case['chunk_min'], case['chunk_max']) for _ in range(case['requests'])]
    hist[-1], new[-1] = case['ctx_max'], case['chunk_max']
    return hist, new


def _valid_lengths(batch, length):
    return [max(2, int(length * (1 - 0.1 * i))) for i in range(batch)]


def _row_lengths(batch, rows):
    return [max(1, int(rows * (1 - 0.05 * i))) for i in range(batch)]


def work(case):
    kind = case['kind']
    if kind == 'step':
        hist, new = _lengths(case)
        nbytes = flops = 0
        T = sum(new)
        for loop in range(LOOPS):
            w = RANK1 if loop == 0 else RANK
            for h, q in zip(hist, new):
                n, m = max(h - WINDOW, 0), min(h, WINDOW)
                pairs = q * m + q * (q + 1) // 2
                nbytes += n * 4 * w + (m + q) * HEADS * HEAD_DIM * 4
                flops += 4 * q * HEADS * n * w + 4 * HEADS * HEAD_DIM * pairs
            nbytes += 2 * HEADS * HEAD_DIM * w * 2 + 3 * T * HEADS * HEAD_DIM * 2     # A, B; q twice, the output
            flops += 4 * T * HEADS * HEAD_DIM * w
        return dict(bytes=nbytes * case['layers'], flops=flops * case['layers'])
    if kind == 'writer':
        T = case['requests'] * case['chunk']
        cols = 2 * RANK1 + 3 * 2 * RANK
        nbytes = cols * HIDDEN * 2 + LOOPS * T * HIDDEN * 2 + T * 2 * (RANK + RANK1) * 2
        return dict(bytes=nbytes * case['layers'], flops=2 * T * HIDDEN * cols * case['layers'])
    if kind == 'rows':
        B, R = case['batch'], case['width']
        rows = sum(_row_lengths(B, case['rows']))
        return dict(bytes=rows * 4 * R + B * case['rows'] + 4 * B * HEADS * R, flops=4 * rows * HEADS * R)
    if kind == 'khop':
        B, L, R = case['batch'], case['length'], case['width']
        pairs = sum(n * (n - 1) // 2 for n in _valid_lengths(B, L))
        size = 2 if case['precision'] == 'bf16' else 4
        # q, dz, z, dq and k, v, dk, dv once each; two products forward, five backward (the scores again among them)
        return dict(bytes=4 * size * B * L * (HEADS + 1) * R + B * L * L, flops=7 * 2 * HEADS * R * pairs)
    B, n = case['batch'], case['chunk']
    w = RANK1 if case['loop'] == 0 else RANK
    rows = case['block0'] + case['block1']
    hist = int(0.8 * B * rows) * HEADS * n
    flops = 7 * (2 * HEAD_DIM * B * HEADS * n * (n + 1) // 2 + 2 * w * hist)
    flops += 12 * B * n * HEADS * HEAD_DIM * w                                        # q A and z B, with backward
    packed = B * rows * 2 * (RANK + RANK1) * 2
    return dict(bytes=packed + B * rows * 4 * w + 9 * B * HEADS * n * HEAD_DIM * 2, flops=flops)


def tolerance(case):
    """bf16 results carry a rounding of 2^-9 each and bf16 softmax weights; the fp32 kind sums up to 2048 products
    in fp32. About four times the distance measured between the path and its float64 reference."""
    if case['kind'] == 'khop' and case['precision'] == 'fp32':
        return dict(rel=1e-5)
    return dict(rel=1e-2)


# ---- inputs ----------------------------------------------------------------------------------------------------

def _gen(seed):
    device = torch.device('cuda:0')
    g = torch.Generator(device=device).manual_seed(int(seed))

    def rnd(*shape, std=1.0, dtype=BF):
        return (torch.randn(*shape, generator=g, device=device, dtype=torch.float32) * std).to(dtype)
    return device, g, rnd


def _rope_table(width):
    """[cos | sin] of the latent angles: the head's frequencies reused round-robin over the width's pairs."""
    inv = 1.0 / (1e6 ** (torch.arange(0, HEAD_DIM, 2, dtype=torch.int64).float() / HEAD_DIM)).cuda()
    pair = torch.arange(width // 2, device='cuda') % inv.shape[0]
    angle = torch.arange(MAX_POSITION, device='cuda').float()[:, None] * inv[pair][None, :]
    return torch.cat((angle.cos(), angle.sin()), -1).to(BF)


def _step_inputs(case, seed):
    device, g, rnd = _gen(seed)
    hist, new = _lengths(case)
    B, T = len(hist), sum(new)
    seq = [h + q for h, q in zip(hist, new)]
    cols = [-(-s // BLOCK) for s in seq]
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=device)

    def tables(first):
        """Random pages for columns ``first[r]``..; page 0 is the null page of the columns before."""
        total = sum(c - f for c, f in zip(cols, first))
        pages = (torch.randperm(total, generator=g, device=device) + 1).to(torch.int32)
        table, used = torch.zeros(B, max(cols), dtype=torch.int32, device=device), 0
        for r in range(B):
            n = cols[r] - first[r]
            table[r, first[r]:cols[r]] = pages[used:used + n]
            used += n
        return table, total + 1

    d = types.SimpleNamespace(hist=hist, new=new, seq=seq, T=T)
    d.table, pool = zip(*(tables([0] * B) for _ in range(2)))                         # widths RANK, RANK1
    d.lat = [[torch.empty(pool[i], 1, BLOCK, 2 * w, dtype=BF, device=device).normal_(generator=g)
              for i, w in enumerate((RANK, RANK1))] for _ in range(case['layers'])]
    # exact caches hold the window's and the step's own tokens; the pages before were given back
    d.ex_table, ex_pool = zip(*(tables([max(0, h - WINDOW) // BLOCK for h in hist]) for _ in range(LOOPS)))
    d.exact = [[rnd(ex_pool[l], BLOCK, HEADS, 2 * HEAD_DIM).transpose(1, 2) for l in range(LOOPS)]
               for _ in range(case['layers'])]
    std = 1 / math.sqrt(HIDDEN)
    d.A = [[rnd(HEADS, HEAD_DIM, RANK1 if l == 0 else RANK, std=std) for l in range(LOOPS)]
           for _ in range(case['layers'])]
    d.B = [[rnd(HEADS, RANK1 if l == 0 else RANK, HEAD_DIM, std=std) for l in range(LOOPS)]
           for _ in range(case['layers'])]
    d.q_pre = [rnd(T, HEADS, HEAD_DIM, std=2.0) for _ in range(LOOPS)]
    d.q_rope = [rnd(T, HEADS, HEAD_DIM, std=2.0) for _ in range(LOOPS)]
    d.positions = torch.tensor([h + i for h, q in zip(hist, new) for i in range(q)], device=device)
    starts = [0]
    for q in new:
        starts.append(starts[-1] + q)
    d.starts, d.qsl, d.seq_lens = starts, i32(starts), i32(seq)
    # the step's own keys and values, as the adapter writes them to the exact caches before it attends
    req = torch.tensor([r for r, q in enumerate(new) for _ in range(q)], device=device)
    d.k_rope, d.v = [], []
    for l in range(LOOPS):
        page = d.ex_table[l][req, d.positions // BLOCK].long()
        row = d.exact[0][l].transpose(1, 2)[page, d.positions % BLOCK]                 # [T, 16, 256]
        for layer in d.exact[1:]:
            layer[l].transpose(1, 2)[page, d.positions % BLOCK] = row
        d.k_rope.append(row[..., :HEAD_DIM].contiguous())
        d.v.append(row[..., HEAD_DIM:].contiguous())
    return d


def _writer_inputs(case, seed):
    device, g, rnd = _gen(seed)
    B, Q = case['requests'], case['chunk']
    d = types.SimpleNamespace(T=B * Q)
    # each request's tokens start a page and fill it in order; a decode token is the last of its request so far
    first = [0 if Q > 1 else 16 * (r % 7) for r in range(B)]
    d.positions = torch.tensor([f + i for f in first for i in range(Q)], device=device)
    d.pages = -(-(max(first) + Q) // BLOCK)
    d.qsl = torch.arange(0, d.T + 1, Q, dtype=torch.int32, device=device)
    d.seq_lens = torch.tensor([f + Q for f in first], dtype=torch.int32, device=device)
    d.table = torch.randperm(B * d.pages, generator=g, device=device).to(torch.int32).view(B, d.pages)
    d.W = [[rnd(2 * (RANK1 if l == 0 else RANK), HIDDEN, std=HIDDEN ** -0.5) for l in range(LOOPS)]
           for _ in range(case['layers'])]
    d.h = [rnd(d.T, HIDDEN) for _ in range(LOOPS)]
    return d


def _rows_inputs(case, seed):
    device, g, rnd = _gen(seed)
    B, N, R = case['batch'], case['rows'], case['width']
    d = types.SimpleNamespace(q=rnd(B, HEADS, R, std=2 * HEAD_DIM ** 0.5 * R ** -0.5), k=rnd(B, N, R), v=rnd(B, N, R))
    lengths = torch.tensor(_row_lengths(B, N), device=device)
    d.mask = torch.arange(N, device=device)[None] < lengths[:, None]
    d.mask[1:2, ::7] = False
    return d


def _khop_inputs(case, seed):
    device, g, rnd = _gen(seed)
    B, L, R = case['batch'], case['length'], case['width']
    leaf = BF if case['precision'] == 'bf16' else torch.float32
    std = 2 * HEAD_DIM ** 0.5 * R ** -0.5
    d = types.SimpleNamespace(q=rnd(B, L, HEADS, R, std=std, dtype=leaf), k=rnd(B, L, R, dtype=leaf),
                              v=rnd(B, L, R, dtype=leaf), dz=rnd(B, L, HEADS, R, dtype=leaf),
                              dlse=rnd(B, HEADS, L, dtype=torch.float32))
    at = torch.arange(L, device=device)
    valid = at[None] < torch.tensor(_valid_lengths(B, L), device=device)[:, None]
    d.mask = valid[:, :, None] & valid[:, None, :] & (at[:, None] > at[None])[None]
    return d


def _mixed_inputs(case, seed):
    device, g, rnd = _gen(seed)
    B, n = case['batch'], case['chunk']
    sizes = (case['block0'], case['block1'])
    w = RANK1 if case['loop'] == 0 else RANK
    d = types.SimpleNamespace()
    d.q, d.k, d.v = (rnd(B, HEADS, n, HEAD_DIM) for _ in range(3))
    d.blocks = [rnd(B, N, 2 * RANK + 2 * RANK1, std=0.5) for N in sizes]
    d.masks = [torch.rand(B, N, generator=g, device=device) < 0.8 for N in sizes]
    d.A, d.B = rnd(HEADS, HEAD_DIM, w, std=HEAD_DIM ** -0.5), rnd(HEADS, w, HEAD_DIM, std=w ** -0.5)
    d.valid = torch.ones(B, n, dtype=torch.bool, device=device)
    d.valid[0, :min(20, n // 2)] = False                                               # left padding of a short row
    pos = sum(sizes) + torch.arange(n, device=device)[None].expand(B, n)
    inv = 1.0 / (1e6 ** (torch.arange(0, HEAD_DIM, 2, device=device).float() / HEAD_DIM))
    ang = torch.cat((pos[..., None] * inv, pos[..., None] * inv), -1)
    d.cos, d.sin = ang.cos(), ang.sin()
    d.dout = rnd(B, HEADS, n, HEAD_DIM) * d.valid[:, None, :, None]                    # padding is never read
    return d


# ---- the passes ------------------------------------------------------------------------------------------------

class _Reader:
    """The layer's latent module as the serving adapter holds it."""

    def __init__(self, A, B):
        self.A, self.B, self.rank, self.rank1, self.loops = A, B, RANK, RANK1, LOOPS

    def readers(self, loop):
        return self.A[loop], self.B[loop], RANK1 if loop == 0 else RANK


class _EngineLatent:
    """The rolling engine's latent module of one layer: readers, the latent query RoPE'd in the tables' precision, and
    the packed row fields ``[K 512 | V 512 | K1 256 | V1 256]``."""
    head_dim = HEAD_DIM

    def __init__(self, A, B):
        self.A, self.B = A, B

    def readers(self, loop):
        return self.A, self.B, RANK1 if loop == 0 else RANK

    def query(self, loop, q, cos, sin):
        idx = torch.arange(self.A.shape[-1] // 2, device=cos.device) % (HEAD_DIM // 2)
        c, s = (torch.cat((t[..., idx], t[..., idx]), -1).unsqueeze(1) for t in (cos, sin))
        x = torch.matmul(q.to(cos.dtype), self.A.to(cos.dtype)[None])
        x1, x2 = x.chunk(2, -1)
        return x * c + torch.cat((-x2, x1), -1) * s

    def fields(self, loop, packed):
        if loop == 0:
            return packed[..., 2 * RANK:2 * RANK + RANK1], packed[..., 2 * RANK + RANK1:]
        return packed[..., :RANK], packed[..., RANK:2 * RANK]


def _captured(fn):
    """``fn`` run once and captured in a HIP graph: the graph and the tensors its replays write."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fn()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fn()
    return dict(graph=graph, out=out, keep=fn)


def _prepare_step(case, seed):
    pkg = importlib.import_module(PKG)
    ops, layer = pkg.s6_ops, pkg.s6_layer
    d = _step_inputs(case, seed)
    cus = pkg._lib.device_cus(0)
    tables = {RANK: _rope_table(RANK), RANK1: _rope_table(RANK1)}
    longest = max(d.seq)
    splits = lambda t: ops.num_kv_splits(longest, t, SPLIT_MAX_TOKENS, cus)
    rows = max(MAX_BATCHED_TOKENS, max(t * splits(t) for t in range(1, SPLIT_MAX_TOKENS + 1)))
    workspace = ops.S6Workspace(HEADS, RANK, rows)
    readers = [_Reader(a, b) for a, b in zip(d.A, d.B)]

    def step():
        ctx = layer.StepContext(d.positions, d.qsl, d.seq_lens, max(d.new), d.T, tables, SCALE, ops.HIP_BACKENDS,
                                workspace, splits(d.T), window=WINDOW, max_seqlen_k=longest)
        out = []
        for loop in range(LOOPS):
            i = 1 if loop == 0 else 0
            for l, sl in enumerate(readers):
                q_lat = ctx.latent_query(sl, loop, d.q_pre[loop])
                out.append(layer.attend(sl, loop, q_lat, d.q_rope[loop], d.k_rope[loop], d.v[loop], d.lat[l][i],
                                        d.table[i], None, None, ctx, (d.exact[l][loop], d.ex_table[loop])))
        return out
    return _captured(step)


def _prepare_writer(case, seed):
    pkg = importlib.import_module(PKG)
    layer = pkg.s6_layer
    d = _writer_inputs(case, seed)
    tables = {RANK: _rope_table(RANK), RANK1: _rope_table(RANK1)}
    sls = []
    for W in d.W:
        lin = [types.SimpleNamespace(weight=w) for w in W]
        sls.append(types.SimpleNamespace(rank=RANK, rank_v=RANK, rank1=RANK1, loops=LOOPS, head_dim=HEAD_DIM,
                                         cand1=lin[0], cand_s=lin[1:]))
    pool = d.table.numel()
    caches = [{w: torch.zeros(pool, 1, BLOCK, 2 * w, dtype=BF, device='cuda') for w in (RANK, RANK1)} for _ in sls]

    def step():
        ctx = layer.StepContext(d.positions, d.qsl, d.seq_lens, case['chunk'], d.T, tables, SCALE,
                                layer.s6_ops.HIP_BACKENDS)
        for sl, cache in zip(sls, caches):
            state = None
            for loop in range(LOOPS):
                state = layer.write_commit(sl, loop, d.h[loop], state, ctx, cache[RANK1 if loop == 0 else RANK],
                                           d.table)
        return [t for cache in caches for t in (cache[RANK], cache[RANK1])]
    return _captured(step)


def _prepare_rows(case, seed):
    hg = importlib.import_module(PKG).history_gemm
    d = _rows_inputs(case, seed)

    def step():
        with torch.no_grad():
            return hg.history_attention(d.q, d.k, d.v, d.mask, SCALE)
    return _captured(step)


def prepare(case, seed):
    if case['kind'] == 'step':
        return _prepare_step(case, seed)
    if case['kind'] == 'writer':
        return _prepare_writer(case, seed)
    if case['kind'] == 'rows':
        return _prepare_rows(case, seed)
    pkg = importlib.import_module(PKG)
    if case['kind'] == 'khop':
        d = _khop_inputs(case, seed)
        leaves = [t.requires_grad_(True) for t in (d.q, d.k, d.v)]

        def train():
            z, lse = pkg.history_gemm.causal_history_gemm(*leaves, d.mask, SCALE, causal=True,
                                                          precision=case['precision'])
            return [z.detach(), lse.detach(), *torch.autograd.grad([z, lse], leaves, [d.dz, d.dlse])]
        return dict(train=train)
    d = _mixed_inputs(case, seed)
    leaves = [t.requires_grad_(True) for t in (d.q, d.k, d.v, *d.blocks, d.A, d.B)]
    sl = _EngineLatent(d.A, d.B)

    def train():
        out = pkg.batched_engine.mixed_attention(sl, case['loop'], d.q, d.k, d.v, d.cos, d.sin, d.valid, d.blocks,
                                                 d.masks)
        return [out.detach(), *torch.autograd.grad(out, leaves, d.dout)]
    return dict(train=train)


def run(state):
    if 'graph' in state:
        state['graph'].replay()
        return state['out']
    return state['train']()


# ---- float64 references ----------------------------------------------------------------------------------------

def _rope64(x, cos, sin):
    x1, x2 = x.chunk(2, -1)
    return x * cos + torch.cat((-x2, x1), -1) * sin


def _exact_step(case, seed):
    d = _step_inputs(case, seed)
    out = []
    for loop in range(LOOPS):
        w, i = (RANK1, 1) if loop == 0 else (RANK, 0)
        table = _rope_table(w)[d.positions].double()
        cos, sin = (t.repeat(1, 2)[:, None] for t in table.chunk(2, -1))
        for l in range(case['layers']):
            q_lat = _rope64(torch.einsum('thd,hdr->thr', d.q_pre[loop].double(), d.A[l][loop].double()), cos, sin)
            got = torch.empty(d.T, HEADS, HEAD_DIM, dtype=torch.float64, device='cuda')
            for r, (h, q) in enumerate(zip(d.hist, d.new)):
                t0, n, first = d.starts[r], max(h - WINDOW, 0), max(h - WINDOW, 0)
                at = torch.arange(n, device='cuda')
                rows = d.lat[l][i][d.table[i][r, at // BLOCK].long(), 0, at % BLOCK].double()
                ex = torch.arange(first, h + q, device='cuda')
                kv = d.exact[l][loop][d.ex_table[loop][r, ex // BLOCK].long(), :, ex % BLOCK].double()   # [m, 16, 256]
                tok = slice(t0, t0 + q)
                s_lat = torch.matmul(q_lat[tok].transpose(0, 1), rows[:, :w].T)                          # [16, q, n]
                s_ex = torch.matmul(d.q_rope[loop][tok].double().transpose(0, 1), kv[..., :HEAD_DIM].permute(1, 2, 0))
                hidden = ex[None] > (h + torch.arange(q, device='cuda'))[:, None]
                s_ex = s_ex.masked_fill(hidden[None], -math.inf)
                p = torch.softmax(torch.cat((s_lat, s_ex), -1) * SCALE, -1)
                o = torch.matmul(torch.matmul(p[..., :n], rows[:, w:]), d.B[l][loop].double())
                o = o + torch.matmul(p[..., n:], kv[..., HEAD_DIM:].transpose(0, 1))
                got[tok] = o.transpose(0, 1)
            out.append(got)
    return out


def _exact_writer(case, seed):
    d = _writer_inputs(case, seed)
    req = torch.arange(d.T, device='cuda') // case['chunk']
    slot = d.table[req, d.positions // BLOCK].long() * BLOCK + d.positions % BLOCK
    out = []
    for W in d.W:
        rows = [h.double() @ w.double().T for h, w in zip(d.h, W)]
        for w, row in ((RANK, rows[1] + rows[2] + rows[3]), (RANK1, rows[0])):
            cos, sin = (t.repeat(1, 2) for t in _rope_table(w)[d.positions].double().chunk(2, -1))
            cache = torch.zeros(d.table.numel() * BLOCK, 2 * w, dtype=torch.float64, device='cuda')
            cache[slot] = torch.cat((_rope64(row[:, :w], cos, sin), row[:, w:]), -1)
            out.append(cache.view(-1, 1, BLOCK, 2 * w))
    return out


def _exact_rows(case, seed):
    d = _rows_inputs(case, seed)
    s = torch.matmul(d.q.double(), d.k.double().transpose(1, 2)) * SCALE
    s = s.masked_fill(~d.mask[:, None], -math.inf)
    return torch.matmul(torch.softmax(s, -1), d.v.double()), torch.logsumexp(s, -1)


def _exact_khop(case, seed):
    d = _khop_inputs(case, seed)
    B, L, R = d.k.shape
    outs = [[] for _ in range(5)]
    for b in range(B):
        k, v, hidden = d.k[b].double(), d.v[b].double(), ~d.mask[b]
        none = hidden.all(-1)
        z, dq = torch.empty(2, L, HEADS, R, dtype=torch.float64, device='cuda')
        lse = torch.empty(HEADS, L, dtype=torch.float64, device='cuda')
        dk, dv = torch.zeros_like(k), torch.zeros_like(v)
        for h in range(HEADS):
            q, dz = d.q[b, :, h].double(), d.dz[b, :, h].double()
            s = ((q @ k.T) * SCALE).masked_fill(hidden, -math.inf)
            lse[h] = torch.logsumexp(s, -1)
            p = torch.exp(s - lse[h].masked_fill(none, 0)[:, None])
            z[:, h] = p @ v
            ds = p * (dz @ v.T - ((dz * z[:, h]).sum(-1) - d.dlse[b, h].double())[:, None]) * SCALE
            dq[:, h] = ds @ k
            dk += ds.T @ q
            dv += p.T @ dz
        for o, t in zip(outs, (z, lse, dq, dk, dv)):
            o.append(t)
    return [torch.stack(o) for o in outs]


def _exact_mixed(case, seed):
    d = _mixed_inputs(case, seed)
    B, n = case['batch'], case['chunk']
    leaf = lambda t: t.double().requires_grad_(True)
    q, k, v, A, Bm = (leaf(t) for t in (d.q, d.k, d.v, d.A, d.B))
    blocks = [leaf(t) for t in d.blocks]
    sl = _EngineLatent(A, Bm)
    cos, sin = d.cos.double(), d.sin.double()
    qr, kr = (_rope64(t, cos[:, None], sin[:, None]) for t in (q, k))
    at = torch.arange(n, device='cuda')
    see = (d.valid[:, None, :] & (at[None, :] <= at[:, None])[None]) | ~d.valid[:, :, None]               # [B, n, n]
    scores = [torch.matmul(qr, kr.transpose(2, 3)).masked_fill(~see[:, None], -math.inf)]
    qc = sl.query(case['loop'], q, cos, sin)
    fields = [sl.fields(case['loop'], b) for b in blocks]
    for (ck, _), m in zip(fields, d.masks):
        s = torch.matmul(qc, ck[:, None].transpose(2, 3))
        scores.append(s.masked_fill(~m[:, None, None], -math.inf))
    p = torch.softmax(torch.cat(scores, -1) * SCALE, -1).split([s.shape[-1] for s in scores], -1)
    z = sum(torch.matmul(pp, cv[:, None]) for pp, (_, cv) in zip(p[1:], fields))
    out = torch.matmul(p[0], v) + torch.matmul(z, Bm[None])
    return [out.detach(), *torch.autograd.grad(out, [q, k, v, *blocks, A, Bm], d.dout.double())]


def exact(case, seed):
    """What ``run`` returns for these inputs, in float64."""
    return dict(step=_exact_step, writer=_exact_writer, rows=_exact_rows, khop=_exact_khop,
                mixed=_exact_mixed)[case['kind']](case, seed)
