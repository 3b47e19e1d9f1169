"""Decode over pages that do not hold whole 16-token blocks (page_size not a
multiple of 16): a block's tokens come from several pages, pages straddle
blocks, and splits given by the caller start inside a block. Lengths end at
page and block edges, tails and spare pages hold NaN; the oracle is the CPU
path."""

from __future__ import annotations

import pytest
import torch

from kernel_lab.kv_cache import random_decode_problem
from oracle import reference as ref
from tests.conftest import DTYPES, decode_parity

pytestmark = pytest.mark.gpu


def _lens(page: int) -> list[int]:
    return [1, 15, 16, 17, page, page + 1, 3 * page + 2, 128, 129, 500, 64 * 16 + 5]


def _check(gpu_ops, lens, hq, hkv, head_dim, page, dtype, splits, **kw):
    q, kv, _, _ = random_decode_problem(lens, hq, hkv, head_dim, page, dtype=dtype, device="cuda", poison=float("nan"),
                                        tail=float("nan"), seed=page + head_dim)
    out = gpu_ops.paged_decode_attention(q, kv.k_cache, kv.v_cache, kv.block_table, kv.seq_lens, num_splits=splits, **kw)
    seq = kv.seq_lens.cpu()
    if "max_seq_len" in kw:
        seq = seq.clamp(max=-(-kw["max_seq_len"] // page) * page)
    want = ref.paged_decode_attention(q.cpu().float(), kv.k_cache.cpu(), kv.v_cache.cpu(), kv.block_table.cpu(), seq)
    decode_parity(out, want, dtype, f"page {page} {hq}/{hkv}/{head_dim} splits {splits}")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("page", [1, 2, 3, 5, 8, 12, 24, 40])
@pytest.mark.parametrize(("hq", "hkv", "head_dim"), [(8, 2, 64), (32, 8, 128), (20, 1, 128), (8, 4, 256), (4, 2, 32), (24, 1, 64)])
def test_small_pages(gpu_ops, dtype, page, hq, hkv, head_dim):
    _check(gpu_ops, _lens(page), hq, hkv, head_dim, page, dtype, None)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("splits", [1, 3, 7, 64, -1])
@pytest.mark.parametrize("page", [1, 5, 8, 20])
def test_small_pages_with_given_splits(gpu_ops, dtype, splits, page):
    _check(gpu_ops, _lens(page), 16, 4, 128, page, dtype, splits)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("page", [1, 3, 8])
def test_small_pages_full_batch_and_one_sequence(gpu_ops, dtype, page):
    _check(gpu_ops, [70 + 5 * b for b in range(40)], 32, 8, 128, page, dtype, None)  # a workgroup per unit
    _check(gpu_ops, [123] * 70, 8, 8, 64, page, dtype, None)  # even lengths
    _check(gpu_ops, [3001], 8, 2, 128, page, dtype, None)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize(("page", "bound"), [(1, 21), (5, 23), (8, 50)])
def test_small_pages_stop_at_max_seq_len(gpu_ops, dtype, page, bound):
    """The bound is counted in the table's pages, not in blocks."""
    _check(gpu_ops, [10, 60, 90, 22], 8, 2, 64, page, dtype, None, max_seq_len=bound)


def test_small_pages_empty_sequences(gpu_ops):
    q, kv, _, _ = random_decode_problem([9, 1, 700], 8, 2, 128, 8, dtype=torch.bfloat16, device="cuda")
    kv.seq_lens[1] = 0
    for splits in (None, 2, -1):
        out = gpu_ops.paged_decode_attention(q, kv.k_cache, kv.v_cache, kv.block_table, kv.seq_lens, num_splits=splits)
        assert (out[1] == 0).all() and torch.isfinite(out).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("splits", [None, 3])
def test_small_pages_infinite_values(gpu_ops, dtype, splits):
    """An infinite value with a positive weight gives an infinite output in its
    head dim and leaves the others alone."""
    q, kv, _, _ = random_decode_problem([700, 40, 5], 8, 2, 128, 8, dtype=dtype, device="cuda")
    for b, tok in ((0, 333), (1, 39), (2, 0)):
        page = int(kv.block_table[b, tok // 8])
        kv.v_cache[page, tok % 8, 0, 7] = float("inf")
        kv.v_cache[page, tok % 8, 1, 100] = -float("inf")
    out = gpu_ops.paged_decode_attention(q, kv.k_cache, kv.v_cache, kv.block_table, kv.seq_lens, num_splits=splits).cpu()
    assert (out[:, :4, 7] == float("inf")).all() and (out[:, 4:, 100] == -float("inf")).all()
    want = ref.paged_decode_attention(q.cpu().float(), kv.k_cache.cpu(), kv.v_cache.cpu(), kv.block_table.cpu(), kv.seq_lens.cpu())
    finite = torch.isfinite(want)
    assert int((~finite).sum()) == 3 * 8
    decode_parity(out.masked_fill(~finite, 0), want.masked_fill(~finite, 0), dtype)
