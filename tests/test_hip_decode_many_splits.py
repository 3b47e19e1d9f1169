"""More given splits than the MFMA kernels' partials reach: a workgroup stores its
heads' rows at 32-bit offsets, so one-token pages cut into some 140,000 splits at
16 heads of 256 dims pass 2 GiB. Either side of that border gives what few splits
give."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(("dtype", "tolerance"), [(torch.float32, 1e-4), (torch.bfloat16, 2**-7)])
@pytest.mark.parametrize("tokens", [139810, 139811])
def test_partials_beyond_two_gib(gpu_ops, dtype, tokens, tolerance):
    """Outputs are about 1, the values' mean. Tolerances: fp32, the merge adds
    139,811 rows to a running sum, each rounded to 2^-24 of it, which walks to
    sqrt(139,811) 2^-24 = 2.2e-5 (times 4); bf16, the output's last place (2^-8)
    twice. A head whose partials were lost is some 1e-2 off."""
    g = torch.Generator(device="cuda").manual_seed(tokens)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    q, k, v = rand(1, 16, 256).to(dtype), rand(tokens, 1, 1, 256).to(dtype), (1 + rand(tokens, 1, 1, 256)).to(dtype)
    table = torch.randperm(tokens, generator=g, device="cuda").to(torch.int32)[None]
    lens = torch.tensor([tokens], dtype=torch.int32, device="cuda")
    few = gpu_ops.paged_decode_attention(q, k, v, table, lens, num_splits=64).float()
    many = gpu_ops.paged_decode_attention(q, k, v, table, lens, num_splits=tokens).float()
    assert (few.mean() - 1).abs() < 0.1
    assert (many - few).abs().max() <= tolerance
