"""The bf16 K-hop kernels at sizes where the library's rule (``hla_s6_khop_multi_query``) takes the multi-query ones for
each part of a call: every test first asks the rule, so that a later change of it cannot move the sizes to the other kernels
unnoticed. Against the float64 oracle with the bars of tests/test_gpu_khop.py."""
import importlib
import math

import numpy as np
import pytest
import torch

from oracle import bf16
from oracle import s6_oracle as O
from s6util import assert_attention_close, assert_lse_close, rel_l2
from test_gpu_khop import assert_grad_close, case
import test_gpu_batched_engine as mixed
import test_gpu_single_history as single

pytestmark = pytest.mark.gpu

hg = importlib.import_module('hybrid-latent-attention_amd.history_gemm')
be = importlib.import_module('hybrid-latent-attention_amd.batched_engine')
ALL = hg.FORWARD | hg.DQ | hg.DKDV


def leaves(*arrays, grad=True):
    return [torch.tensor(x, device='cuda').to(torch.bfloat16).requires_grad_(grad) for x in arrays]


def cotangents(shape, seed):
    rng = np.random.default_rng(seed)
    B, Lq = shape[:2]
    return (bf16.round_bf16(rng.standard_normal(shape).astype(np.float32)),
            rng.standard_normal((B, 16, Lq)).astype(np.float32))


def gradients(z, lse, inputs, dz, dlse):
    return torch.autograd.grad([z, lse], inputs, [torch.tensor(dz, device='cuda').to(z.dtype),
                                                  torch.tensor(dlse, device='cuda')])


def assert_oracle(q, k, v, mask, scale, got, dz, dlse, what, rows):
    """z, lse, dq, dk, dv of the batch rows ``rows`` (a row's results depend on that row alone)."""
    q, k, v, mask, dz, dlse = (np.asarray(x)[rows] for x in (q, k, v, mask, dz, dlse))
    z, lse, *grads = (t.detach()[rows].float().cpu().numpy() for t in got)
    zo, lo = O.causal_history(q, k, v, mask, scale)
    assert_attention_close(z, zo, f'z ({what})')
    assert_lse_close(lse, lo)
    for name, g, want in zip(('dq', 'dk', 'dv'), grads, O.causal_history_backward(q, k, v, mask, scale, lo, dz, dlse)):
        assert_grad_close(g, want, f'{name} ({what})')


@pytest.mark.parametrize('R', [256, 512])
@pytest.mark.parametrize('N', [784, 785])
def test_one_mask_row_and_a_copy_per_query(R, N):
    """One mask row for all queries (dk / dv cut over all tokens in two shares, tiles side by side) and its copy per query
    (shares of each tile's own tokens), with whole and with padded mask rows: forward and dq bitwise alike, dk / dv alike but
    for the order of fp32 sums, everything as the oracle."""
    B, Lq, scale = 13, 80, 0.06
    q, k, v, _ = case(R + N, B, Lq, N, R, 'any')
    rows = np.random.default_rng(N).random((B, N)) < 0.6
    rows[1] = False
    rows[-1, N // 3:] = False
    dz, dlse = cotangents(q.shape, R)
    dlse[1] = 0                                                # (lse = -inf there)
    out = []
    for copied in (False, True):
        mt = torch.tensor(rows, device='cuda')[:, None].expand(B, Lq, N)
        mt = mt.contiguous() if copied else mt
        assert hg._multi(B, Lq, N, R, mt.stride(1)) == ALL
        print(f'case copied={copied} R={R} N={N}', flush=True)
        x = leaves(q, k, v)
        z, lse = hg.causal_history_gemm(*x, mt, scale, precision='bf16')
        out.append((z, lse, *gradients(z, lse, x, dz, dlse)))
    assert all(torch.equal(a, b) for a, b in zip(out[0][:3], out[1][:3]))
    assert not out[0][2][1].any() and not out[0][3][1].any()
    for a, b in zip(out[0][3:], out[1][3:]):
        assert_grad_close(a.float().cpu().numpy(), b.float().cpu().numpy(), 'one row against its copies')
    mask = np.broadcast_to(rows[:, None], (B, Lq, N))
    assert_oracle(q, k, v, mask, scale, out[0], dz, dlse, 'one row', [0, B - 1])


@pytest.mark.parametrize('R', [256, 512])
@pytest.mark.parametrize('N', [784, 785])
def test_no_mask_through_the_c_abi(R, N):
    """Every key below the bound visible (the kernels' forms without a mask), whole and ragged key counts, dk / dv in three
    shares and in one."""
    B, Lq, scale, lib = 13, 80, 0.05, hg._lib
    assert hg._multi(B, Lq, N, R, 0) == ALL
    q, k, v, _ = case(N - R, B, Lq, N, R, 'any')
    dz, dlse = cotangents(q.shape, N)
    qt, kt, vt, dzt = leaves(q, k, v, dz, grad=False)
    dlt = torch.tensor(dlse, device='cuda')
    P, st = lib.ptr, lib.stream(qt.device)
    print(f'case no mask R={R} N={N}', flush=True)
    bound = torch.empty(B * Lq, dtype=torch.int32, device='cuda')
    lib.call('hla_s6_khop_bounds', None, 0, 0, B, Lq, N, P(bound), st)
    z = torch.empty(B, Lq, 16, R, dtype=torch.bfloat16, device='cuda')
    lse, delta = (torch.empty(B, 16, Lq, device='cuda') for _ in range(2))
    inputs = (P(qt), *qt.stride()[:3], P(kt), *kt.stride()[:2], P(vt), *vt.stride()[:2], None, 0, 0, P(bound), B, Lq, N, 16,
              R, scale)
    lib.call('hla_s6_khop_forward', *inputs, P(z), *z.stride()[:3], P(lse), st)
    out = {}
    for splits in (1, 3):
        dq, dk, dv = torch.empty(B, Lq, 16, R, device='cuda'), *(torch.empty(B, N, R, device='cuda') for _ in range(2))
        ws = torch.empty(max(1, lib.load().hla_s6_khop_backward_workspace(B, Lq, N, R, splits)), device='cuda')
        lib.call('hla_s6_khop_backward', *inputs, P(z), *z.stride()[:3], P(lse), P(dzt), *dzt.stride()[:3], P(dlt), P(delta),
                 P(dq), *dq.stride()[:3], P(dk), *dk.stride()[:2], P(dv), *dv.stride()[:2], splits, P(ws), ws.numel(), 0, st)
        out[splits] = (dq, dk, dv)
    for name, a, b in zip(('dq', 'dk', 'dv'), out[1], out[3]):
        assert_grad_close(a.cpu().numpy(), b.cpu().numpy(), f'{name} in one share')
    assert_oracle(q, k, v, np.ones((B, Lq, N), bool), scale, (z, lse, *out[3]), dz, dlse, 'no mask', [0, B - 1])


def test_width_256_forward_with_one_and_two_tokens_per_wave():
    """Two tokens per wave when the grid has more 8-token workgroups than the device has CUs, else one: batch row 0 of
    33 x 64 queries and of 16 x 64 queries over 784 keys."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    R, Lq, N, scale = 256, 64, 784, 1 / 16
    B = -(-8 * (cus + 8) // Lq)
    q, k, v, mask = case(5, B, Lq, N, R, 'any')
    x, mt = leaves(q, k, v, grad=False), torch.tensor(mask, device='cuda')
    zo, lo = O.causal_history(q[:1], k[:1], v[:1], mask[:1], scale)
    for rows in (B, 16):
        assert hg._multi(rows, Lq, N, R, N) & hg.FORWARD and (rows * Lq > 8 * cus) == (rows == B)
        z, lse = hg.causal_history_gemm(*(t[:rows] for t in x), mt[:rows], scale, precision='bf16')
        assert_attention_close(z[:1].float().cpu().numpy(), zo, f'z ({rows} rows)')
        assert_lse_close(lse[:1].cpu().numpy(), lo)


@pytest.mark.parametrize('R', [256, 512])
@pytest.mark.parametrize('B,Lq,N', [(4, 2, 784), (1, 5, 2047), (3, 33, 785), (2, 1, 769)])
def test_few_queries_over_many_keys(R, B, Lq, N):
    """dq over key ranges with partials, forward on the 32-key kernel; bf16 gradients are the rounded fp32 ones."""
    assert hg._multi(B, Lq, N, R, N) & (hg.FORWARD | hg.DQ) == hg.DQ
    q, k, v, mask = case(R + N, B, Lq, N, R, 'any' if Lq > 1 else 'khop')
    dz, dlse = cotangents(q.shape, B)
    dlse = np.where(mask.any(-1)[:, None], dlse, 0).astype(np.float32)   # (lse = -inf there)
    mt, scale, grads = torch.tensor(mask, device='cuda'), 0.07, {}
    for dt in (torch.float32, torch.bfloat16):
        x = [torch.tensor(a, device='cuda').to(torch.bfloat16).to(dt).requires_grad_(True) for a in (q, k, v)]
        z, lse = hg.causal_history_gemm(*x, mt, scale, precision='bf16')
        grads[dt] = gradients(z, lse, x, dz, dlse)
    for name, g32, g16 in zip('qkv', grads[torch.float32], grads[torch.bfloat16]):
        assert torch.equal(g32.to(torch.bfloat16).view(torch.int16), g16.view(torch.int16)), name
    assert_oracle(q, k, v, mask, scale, (z, lse, *grads[torch.float32]), dz, dlse, 'few queries', slice(None))


@pytest.mark.parametrize('R,B,N', [(256, 18, 785), (512, 18, 785), (256, 3, 784), (512, 3, 2047)])
def test_single_query_gradients_over_many_keys(R, B, N):
    """``history_attention``'s backward at key counts on and off 16: dq over key ranges, dk / dv of one query per row."""
    parts = hg._multi(B, 1, N, R, N)
    assert parts & hg.DQ and bool(parts & hg.DKDV) == (R == 256 and B == 18)
    q, k, v, mask = single.case(R + N, B, N, R, 'any')
    rng = np.random.default_rng(B)
    dz = bf16.round_bf16(rng.standard_normal((B, 16, R)).astype(np.float32))
    dlse = rng.standard_normal((B, 16)).astype(np.float32)
    got = single.run(q, k, v, mask, 0.08, dz=dz, dlse=dlse)
    z, lse = single.check_forward(got, q, k, v, mask, 0.08)
    for name, want in zip(('dq', 'dk', 'dv'), O.single_history_backward(q, k, v, mask, 0.08, lse, dz, dlse)):
        assert_grad_close(got[name], want, name)


@pytest.mark.parametrize('loop', [0, 2])
def test_joint_attention_over_a_ragged_block(loop):
    """A chunk of 80 queries over blocks of 785 and 80 rows: output and gradients of two batch rows."""
    B, n, sizes, rows = 13, 80, (785, 80), [0, 12]
    assert hg._multi(B, n, sizes[0], mixed.RANK1 if loop == 0 else mixed.RANK, 0) == ALL
    sl, q, k, v, cos, sin, valid, blocks, masks = mixed.make_case(loop, B, n, sizes, loop, 'left')
    x = [t.clone().requires_grad_(True) for t in (q, k, v, *blocks)]
    out = be.mixed_attention(sl, loop, *x[:3], cos, sin, valid, tuple(x[3:]), tuple(masks))
    g = torch.randn(out.shape, generator=torch.Generator(device='cuda').manual_seed(5), device='cuda')
    g = g * valid[:, None, :, None]
    grads = torch.autograd.grad(out.float(), x, g)
    f64 = lambda t: t.detach()[rows].double().cpu().numpy()
    whole = lambda t: t.detach().double().cpu().numpy()
    fields = [sl.fields(loop, f64(blk)) for blk in blocks]
    args = (f64(q), f64(k), f64(v), f64(cos), f64(sin), valid[rows].cpu().numpy(), [a for a, _ in fields],
            [b for _, b in fields], [m[rows].cpu().numpy() for m in masks], whole(sl.A[loop]), whole(sl.B[loop]),
            1 / math.sqrt(mixed.HD))
    seen = valid[rows].cpu().numpy()
    assert_attention_close(f64(out).transpose(0, 2, 1, 3)[seen], O.mixed_attention(*args).transpose(0, 2, 1, 3)[seen], 'out')
    want = O.mixed_attention_backward(*args, f64(g))
    for name, a in zip('qkv', grads):
        assert rel_l2(f64(a), want[name]) <= 2e-2, name
    for i, a in enumerate(grads[3:]):
        for name, field in zip(('hist_k', 'hist_v'), sl.fields(loop, f64(a))):
            assert rel_l2(field, want[name][i]) <= 2e-2, (name, i)


@pytest.mark.parametrize('R', [256, 512])
@pytest.mark.parametrize('B,Lq,N', [(4, 301, 301), (13, 80, 801)])
def test_causal_rows(R, B, Lq, N):
    """Causal rows of ragged length, more and as many keys as queries, repeatable bit for bit."""
    assert hg._multi(B, Lq, N, R, N) & (hg.DQ | hg.DKDV) and hg._multi(B, Lq, N, 512, N) & hg.DKDV
    q, k, v, mask = case(R + Lq, B, Lq, N, R, 'benchmark' if Lq == N else 'khop')
    dz, dlse = cotangents(q.shape, Lq)
    dlse = np.where(mask.any(-1)[:, None], dlse, 0).astype(np.float32)
    mt, scale, outs = torch.tensor(mask, device='cuda'), 1 / math.sqrt(128), []
    for _ in range(2):
        x = leaves(q, k, v)
        z, lse = hg.causal_history_gemm(*x, mt, scale, precision='bf16')
        outs.append((z, lse, *gradients(z, lse, x, dz, dlse)))
    assert all(torch.equal(a, b) for a, b in zip(*outs))
    assert_oracle(q, k, v, mask, scale, outs[0], dz, dlse, 'causal', [0, B - 1])


@pytest.mark.parametrize('R,B,L,shares', [(256, 128, 129, 1), (512, 128, 129, 1), (256, 18, 257, 6), (512, 6, 331, 14)])
def test_causal_rows_in_one_share_and_in_several(R, B, L, shares):
    """Many batch rows: a tile's queries in one workgroup, dk / dv written without partials; and several shares."""
    q, k, v, mask = case(R, B, L, L, R, 'benchmark')
    mt = torch.tensor(mask, device='cuda')
    assert hg._multi(B, L, L, R, L) & hg.DKDV and hg._shares(B, L, L, R, L, mt.device) == shares
    dz, dlse = cotangents(q.shape, L)
    dlse = np.where(mask.any(-1)[:, None], dlse, 0).astype(np.float32)
    x = leaves(q, k, v)
    z, lse = hg.causal_history_gemm(*x, mt, 0.08, precision='bf16')
    assert_oracle(q, k, v, mask, 0.08, (z, lse, *gradients(z, lse, x, dz, dlse)), dz, dlse, 'shares', [0, 5, B - 1])


@pytest.mark.parametrize('R', [256, 512])
@pytest.mark.parametrize('B,Lq,N', [(13, 80, 785), (8, 256, 256)])
def test_largest_weights_are_exact_at_ragged_and_short_key_ranges(R, B, Lq, N):
    """Scores of standard deviation 3, whose largest weight decides most of z: relative to the true maximum so far that weight
    is 1, exact in bf16, and what is left is the rounding of z (uniform in a bf16 step: 2^-9 / sqrt(3) of the step's top, at
    most 1.7e-3 of the norm) and of the small weights (half of that at most: together 1.9e-3). Relative to a maximum raised
    late the largest weight is rounded like any other (2.1e-3)."""
    assert hg._multi(B, Lq, N, R, 0) & hg.FORWARD
    g = torch.Generator(device='cuda').manual_seed(N)
    q, k, v = (torch.randn(*s, generator=g, device='cuda').to(torch.bfloat16) for s in ((B, Lq, 16, R), (B, N, R), (B, N, R)))
    mt = torch.ones(B, N, dtype=torch.bool, device='cuda')[:, None].expand(B, Lq, N)
    z, _ = hg.causal_history_gemm(q, k, v, mt, 3 / math.sqrt(R), precision='bf16')
    for b in (0, B - 1):
        s = q[b].double().view(-1, R) @ k[b].double().T * (3 / math.sqrt(R))
        want = torch.softmax(s, -1) @ v[b].double()
        err = float((z[b].double().view(-1, R) - want).norm() / want.norm())
        assert err <= 1.9e-3, err
