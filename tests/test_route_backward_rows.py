"""The row kernel of the route's and the dense attention's backward.

Calls the C entry point on both of its forms, runs of four columns and single
ones (chosen by the column count, the pitches and the alignment of the
pointers), at the edges of the columns a lane holds, with and without the
causal bound, against the same operation in 64 bits.
"""

from __future__ import annotations

import pytest
import torch

from double_attention import _lib

pytestmark = pytest.mark.gpu


def _rows(rows, atoms, period, *, shift=0, pitch=0, out_pitch=0, silu=False, dtype=torch.bfloat16):
    """Run the entry on `shift` floats past an aligned start, rows `pitch`
    apart (0: atoms rounded up to four); returns outputs and 64-bit results."""

    g = torch.Generator().manual_seed(atoms + rows)
    d = torch.device("cuda:0")
    ld_in = pitch or (atoms + 3) // 4 * 4
    ld_out = out_pitch or ld_in
    beta = torch.tensor([3.0, 9.0])
    beta_period = max(1, rows // 3)

    def placed(fill):
        buf = torch.full((shift + rows * ld_in,), float("nan"))
        view = buf[shift:].view(rows, ld_in)
        view[:, :atoms] = fill
        if period:   # what lies past a row's last column is never used
            past = torch.arange(atoms)[None] > (torch.arange(rows) % period)[:, None]
            view[:, :atoms][past] = float("nan")
        return buf.to(d)

    l = torch.rand(rows, atoms, generator=g) * 2 - 1
    dw = torch.randn(rows, atoms, generator=g)
    ld, gd, bd = placed(l), placed(dw), beta.to(d)
    code = _lib.DA_BF16 if dtype == torch.bfloat16 else _lib.DA_F16
    outs = [torch.full((shift + rows * ld_out,), float("nan"), dtype=dtype, device=d) for _ in range(2)]
    dbeta = torch.full((rows,), float("nan"), device=d)
    _lib.check(
        _lib.get().da_dictionary_route_backward_rows(
            ld.data_ptr() + 4 * shift, gd.data_ptr() + 4 * shift, rows, atoms, period, ld_in,
            bd.data_ptr(), _lib.DA_F32, 0.0, 2, beta_period, _lib.DA_ROUTE_SILU_LOGITS if silu else 0, 1.0, 1.0, 1e-6,
            outs[0].data_ptr() + 2 * shift, outs[1].data_ptr() + 2 * shift, ld_out, code, dbeta.data_ptr(),
            torch.cuda.current_stream().cuda_stream,
        ),
        "route backward rows",
    )
    torch.cuda.synchronize()
    got = []
    for o in outs:
        view = o[shift:].view(rows, ld_out)
        assert view[:, atoms:].isnan().all() and o[:shift].isnan().all()   # nothing written past the columns
        got.append(view[:, :atoms].double().cpu())

    r = torch.arange(rows)
    b = beta.double()[(r // beta_period) % 2][:, None]
    x = l.double().requires_grad_(True)
    c = 2 * torch.nn.functional.silu(x) if silu else x
    scores = b * c
    if period:
        scores = scores.masked_fill(torch.arange(atoms)[None] > (r % period)[:, None], -torch.inf)
    w = torch.softmax(scores, dim=-1)
    (dl,) = torch.autograd.grad((w * dw.double()).sum(), x)
    db = (w * (dw.double() - (w * dw.double()).sum(-1, keepdim=True)) * c).sum(-1).detach()
    # fp32: exponents reach 2 * 9 * 2 (SiLU doubles the logits), so a weight is off
    # by up to 1e-5 of itself; the gradient takes that from both terms of
    # dw - <w, dw>, times beta and the SiLU's slope (at most 2.2).
    seen = dw if not period else dw.masked_fill(torch.arange(atoms)[None] > (r % period)[:, None], 0.0)
    w = w.detach()
    off_w = 1e-5 * w
    off_dl = 2 * 1e-5 * w * b * seen.abs().amax(-1, keepdim=True).double() * (2.2 if silu else 1)
    return got, (dl, w), (off_dl, off_w), dbeta.double().cpu(), db


def _check(result, dtype) -> None:
    got, expected, off, dbeta, db = result
    unit = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)   # half a unit in the last place, relative
    for a, b, o in zip(got, expected, off):
        # The output's rounding (fp16: or half its smallest value) on top.
        bar = b.abs() * unit * 1.01 + o + 2.0 ** -25
        assert ((a - b).abs() <= bar).all(), ((a - b).abs() - bar).max()
    assert (dbeta - db).abs().max() <= 1e-5 * max(1.0, db.abs().max())


@pytest.mark.parametrize("period", [0, 37])
@pytest.mark.parametrize("atoms", [1, 4, 64, 252, 256, 260, 511, 512, 516, 1024, 1028, 2044, 2052, 4096, 4100, 8192,
                                   8196, 16384, 16388])
def test_route_backward_rows_columns(atoms, period) -> None:
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    print(f"[route backward rows] {atoms} columns, period {period}", flush=True)
    dtype = torch.bfloat16 if atoms % 8 else torch.float16
    _check(_rows(75, atoms, period, dtype=dtype), dtype)


@pytest.mark.parametrize("layout", [
    {"shift": 1},                       # misaligned pointers
    {"shift": 4},                       # aligned again
    {"pitch": 530}, {"pitch": 532},     # pitches that are and are not multiples of four
    {"out_pitch": 514}, {"out_pitch": 516},
    {"silu": True}, {"silu": True, "shift": 3},
])
@pytest.mark.parametrize("atoms", [512, 5000])
@pytest.mark.parametrize("period", [0, 37])
def test_route_backward_rows_layouts(layout, atoms, period) -> None:
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    print(f"[route backward rows] {layout} {atoms} columns, period {period}", flush=True)
    layout = {k: v + (5000 - 512 if atoms == 5000 else 0) if "pitch" in k else v for k, v in layout.items()}
    _check(_rows(41, atoms, period, **layout), torch.bfloat16)
