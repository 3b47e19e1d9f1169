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


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("hidden", [64, 100, 128, 1024, 1500])
def test_two_strides_of_leading_dimensions(gpu_ops, dtype, hidden):
    """Leading dimensions that need two strides are read in place (one part of
    a fused projection, a transposed pair), more of them from a copy."""
    base = torch.randn(5, 7, 6, hidden + 12, device="cuda").to(dtype)
    w = (1 + 0.1 * torch.randn(hidden, device="cuda")).to(dtype)
    views = {
        "part of a projection": base[0, :, 1:4, :hidden],
        "shifted": base[0, :, 1:4, 3 : hidden + 3],
        "transposed": base[1].transpose(0, 1)[..., :hidden],
        "one inner row": base[:, :, 2:3, :hidden],
        "groups that nest": base[:, :, :4, :hidden],
        "three strides": base[::2, :5, :4, :hidden],
        "expanded": base[:1, 0, :, :hidden].expand(3, 6, hidden),
    }
    for name, x in views.items():
        out = torch.empty(x.shape, dtype=dtype, device="cuda")
        torch.ops.kernel_lab.rms_norm(out, x, w, 1e-6)
        want = ref.rms_norm(x.cpu(), w.cpu())
        torch.testing.assert_close(out.cpu(), want, **tolerance(dtype), msg=lambda m: f"{name}: {m}")
        res = torch.randn(x.shape, device="cuda").to(dtype)
        got, new = gpu_ops.fused_add_rms_norm(x, res, w)
        want, want_res = ref.fused_add_rms_norm(x.cpu(), res.cpu(), w.cpu())
        assert torch.equal(new.cpu(), want_res), name
        torch.testing.assert_close(got.cpu(), want, **tolerance(dtype), msg=lambda m: f"{name}: {m}")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("hidden", [5, 128, 1000, 1001, 4096, 40000, 100000])
def test_functional_form_equals_the_in_place_one(gpu_ops, dtype, hidden):
    x, r = (torch.randn(3, hidden, device="cuda").to(dtype) for _ in range(2))
    w = (1 + 0.1 * torch.randn(hidden, device="cuda")).to(dtype)
    x0, r0 = x.clone(), r.clone()
    out, new = gpu_ops.fused_add_rms_norm(x, r, w)
    assert torch.equal(x, x0) and torch.equal(r, r0)
    inplace = r.clone()
    want = gpu_ops.fused_add_rms_norm_(x, inplace, w)
    assert torch.equal(out, want) and torch.equal(new, inplace)
    wide = torch.randn(hidden, 3, device="cuda").to(dtype).t()  # a residual with other strides
    out, new = gpu_ops.fused_add_rms_norm(x, wide, w)
    want, want_res = ref.fused_add_rms_norm(x.cpu(), wide.cpu(), w.cpu())
    assert new.is_contiguous() and torch.equal(new.cpu(), want_res)
    torch.testing.assert_close(out.cpu(), want, **tolerance(dtype))


def test_functional_form_keeps_what_a_clone_carries(gpu_ops):
    """A residual with a history is cloned as before, so the new residual
    stays connected to it."""
    x, w = torch.randn(2, 64, device="cuda"), torch.ones(64, device="cuda")
    r = torch.randn(2, 64, device="cuda", requires_grad=True)
    _, new = gpu_ops.fused_add_rms_norm(x, r, w)
    assert new.requires_grad
    with torch.no_grad():
        assert not gpu_ops.fused_add_rms_norm(x, r, w)[1].requires_grad
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(r.detach(), torch.ones_like(r))
        _, new = gpu_ops.fused_add_rms_norm(x, dual, w)
        assert torch.autograd.forward_ad.unpack_dual(new).tangent is not None


def test_functional_form_compiles(gpu_ops):
    x, r, w = torch.randn(4, 256, device="cuda"), torch.randn(4, 256, device="cuda"), torch.ones(256, device="cuda")
    fn = torch.compile(lambda a, b, c: gpu_ops.fused_add_rms_norm(a, b, c), fullgraph=True, backend="aot_eager")
    for got, want in zip(fn(x, r, w), gpu_ops.fused_add_rms_norm(x, r, w), strict=True):
        assert torch.equal(got, want)
