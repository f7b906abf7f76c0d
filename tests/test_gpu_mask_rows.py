"""``history_gemm._mask_bytes``: the mask rows that the multi-query kernels read in whole 16-byte groups and the key
bounds, over every layout a caller may pass (``hla_s6_khop_mask_rows`` where the mask has another form)."""
import importlib

import pytest
import torch

pytestmark = pytest.mark.gpu

hg = importlib.import_module('hybrid-latent-attention_amd.history_gemm')


def layouts(B, Lq, N):
    g = torch.Generator(device='cuda').manual_seed(B * 1000 + Lq * 100 + N)
    rnd = lambda *s: torch.rand(*s, generator=g, device='cuda') < 0.2
    yield 'contiguous', rnd(B, Lq, N)
    yield 'expanded over queries', rnd(B, N)[:, None].expand(B, Lq, N)
    yield 'expanded over the batch', rnd(1, Lq, N).expand(B, Lq, N)
    for off in (1, 2, 3, 16):
        yield f'columns from {off}', rnd(B, Lq, N + off)[..., off:]
    yield 'leading columns of wider rows', rnd(B, Lq, -(-N // 16) * 16 + 16)[..., :N]
    yield 'transposed', rnd(B, N, Lq).transpose(1, 2)
    yield 'every second query', rnd(B, 2 * Lq, N)[:, ::2]
    yield 'nothing visible', torch.zeros(B, Lq, N, dtype=torch.bool, device='cuda')
    yield 'integers', rnd(B, Lq, N).int() * 512


@pytest.mark.parametrize('N', [769, 783, 784, 785, 831, 1023, 2100])
@pytest.mark.parametrize('B,Lq', [(1, 1), (1, 3), (3, 1), (2, 70)])
def test_rows_are_whole_groups_with_the_mask_and_its_bounds(B, Lq, N):
    for name, mask in layouts(B, Lq, N):
        got, bound = hg._mask_bytes(mask, B, Lq, N, mask.device, 512)
        want = mask.bool()
        assert got.dtype == torch.uint8 and got.shape[:2] == (B, Lq), name
        assert torch.equal(got[..., :N] != 0, want), name
        assert got.data_ptr() % 16 == 0 and got.stride(0) % 16 == 0 and got.stride(1) % 16 == 0, name
        last = got.storage_offset() + (B - 1) * got.stride(0) + (Lq - 1) * got.stride(1)
        assert last + -(-N // 16) * 16 <= got.untyped_storage().nbytes(), name
        keys = torch.arange(1, N + 1, device='cuda')
        assert torch.equal(bound.view(B, Lq).long(), (want * keys).amax(-1)), name
        same, plain = hg._mask_bytes(mask, B, Lq, N, mask.device)          # the mask's own rows: bounds alone
        assert torch.equal(same != 0, want) and torch.equal(plain, bound), name
