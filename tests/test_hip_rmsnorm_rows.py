"""RMSNorm over narrow rows (a few lanes per row) and over rows of any width and
address, at the edges of the packs (8 or 4 elements), of the lanes per row and
of the kernels' ranges, against the CPU oracle. The operands sit inside larger
buffers whose neighbouring elements must not change."""

from __future__ import annotations

import pytest
import torch

from oracle import reference as ref
from tests.conftest import DTYPES, tolerance

pytestmark = pytest.mark.gpu

WIDTHS = [1, 3, 4, 7, 8, 9, 12, 31, 32, 33, 40, 63, 64, 65, 100, 127, 128, 129, 255, 256, 257, 511, 512, 513, 1000, 1023,
          1024, 1025, 1028, 2049, 4100, 5003, 8191, 16384, 16385, 33001]


def _inside(t: torch.Tensor, shift: int) -> tuple[torch.Tensor, torch.Tensor]:
    """t at `shift` elements into a buffer of sevens, and the buffer."""
    buf = torch.full((t.numel() + 64,), 7.0, dtype=t.dtype, device="cuda")
    view = buf[shift : shift + t.numel()].view(t.shape)
    view.copy_(t)
    return view, buf


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("shift", [0, 1, 6])
def test_narrow_and_ragged_rows(gpu_ops, dtype, fused, shift):
    for hidden in WIDTHS:
        rows = 67 if hidden < 300 else 5 if hidden < 4000 else 2
        gen = torch.Generator().manual_seed(hidden)
        x, r = (torch.randn(rows, hidden, generator=gen).to(dtype) for _ in range(2))
        w = (1 + 0.1 * torch.randn(hidden, generator=gen)).to(dtype)
        dx, _ = _inside(x.cuda(), shift)
        dw, _ = _inside(w.cuda(), shift)
        out, out_buf = _inside(torch.zeros_like(x).cuda(), shift)
        if fused:
            dr, r_buf = _inside(r.cuda(), shift)
            torch.ops.kernel_lab.fused_add_rms_norm(out, dx, dr, dw, 1e-6)
            want, res = ref.fused_add_rms_norm(x, r, w)
            assert torch.equal(dr.cpu(), res), hidden
            buffers = (out_buf, r_buf)
        else:
            torch.ops.kernel_lab.rms_norm(out, dx, dw, 1e-6)
            want = ref.rms_norm(x, w)
            buffers = (out_buf,)
        torch.testing.assert_close(out.cpu(), want, **tolerance(dtype), msg=lambda m: f"hidden {hidden}: {m}")
        for buf in buffers:
            edge = torch.cat([buf[:shift], buf[shift + rows * hidden :]])
            assert (edge == 7).all(), hidden


@pytest.mark.parametrize("rows", [1, 15, 16, 17, 63, 64, 65, 1000])
def test_last_workgroup_of_narrow_rows(gpu_ops, rows):
    for hidden in (32, 64, 128, 256, 512, 1024):
        x = torch.randn(rows, hidden, device="cuda", dtype=torch.bfloat16)
        w = torch.ones(hidden, device="cuda", dtype=torch.bfloat16)
        torch.testing.assert_close(gpu_ops.rms_norm(x, w).cpu(), ref.rms_norm(x.cpu(), w.cpu()), **tolerance(torch.bfloat16))
