"""The eight-wave route kernel (256- and 512-wide rows, plain softmax).

Sizes where its tiling can go wrong: edges of the 32- and 64-row workgroups and
of the rules between them, dictionaries that end
inside, on and past a 32-atom window, fixed and per-row exponent references,
strided and in-place rows, a log beta on the device; against the same operation
in 64 bits.
"""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from double_attention import _lib

pytestmark = pytest.mark.gpu

CODES = {torch.float16: _lib.DA_F16, torch.bfloat16: _lib.DA_BF16}


@pytest.mark.parametrize("case", [
    # rows, width, atoms, dtype, out dtype, beta, normalize input, output
    (1, 256, 1, torch.bfloat16, torch.float16, 4.0, True, True),
    (33, 256, 33, torch.bfloat16, torch.bfloat16, -6.0, True, True),
    (95, 256, 160, torch.float16, torch.float16, 40.0, True, True),       # row maxima first
    (8192, 256, 512, torch.bfloat16, torch.float16, 8.0, True, True),
    (16320, 256, 65, torch.bfloat16, torch.bfloat16, 9.0, True, False),   # the most rows it takes
    (16321, 256, 65, torch.bfloat16, torch.bfloat16, 9.0, True, False),   # the general kernel
    (12000, 256, 31, torch.bfloat16, torch.float16, 50.0, True, True),
    (31, 512, 512, torch.bfloat16, torch.float16, 8.0, True, True),
    (64, 512, 97, torch.float16, torch.float16, -20.0, False, True),
    (65, 512, 64, torch.bfloat16, torch.bfloat16, 1.0, False, False),     # bf16 keys
    (8192, 512, 95, torch.bfloat16, torch.float16, 8.0, True, True),      # the most 32-row workgroups
    (8193, 512, 96, torch.bfloat16, torch.float16, 8.0, True, True),
    (16383, 512, 1, torch.bfloat16, torch.float16, 4.0, True, True),
    (16385, 512, 1535, torch.bfloat16, torch.float16, 8.0, True, True),
    (16400, 512, 33, torch.float16, torch.float16, 30.0, True, True),
    # Row maxima that move from tile to tile, each kind of workgroup.
    (300, 256, 700, torch.bfloat16, torch.float16, 60.0, True, True),
    (300, 512, 700, torch.bfloat16, torch.bfloat16, -40.0, True, True),
    (8200, 512, 161, torch.float16, torch.float16, 25.0, True, False),
])
@pytest.mark.parametrize("in_place", [False, True])
def test_route_tile(case, in_place, log_beta=False) -> None:
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    rows, width, atoms, dtype, out_dtype, beta, norm_in, norm_out = case
    print(f"[route tile] {case} in place {in_place}", flush=True)
    g = torch.Generator().manual_seed(rows + atoms)
    key_dtype = torch.float16 if norm_in else dtype
    x = (torch.randn(rows, width, generator=g) * (1.0 if norm_in else width ** -0.5)).to(dtype)
    key = F.normalize(torch.randn(atoms, width, generator=g), dim=-1).to(key_dtype)
    value = F.normalize(torch.randn(atoms, width, generator=g), dim=-1).half()
    # Rows near an atom, so that the weights differ.
    x = (x.float() + 2 * key[torch.arange(rows) % atoms].float() * x.float().norm(dim=-1, keepdim=True)).to(dtype)

    padded = (atoms + 63) // 64 * 64
    key_t = torch.zeros(padded, width, dtype=key_dtype)
    key_t[:atoms] = key
    tiles = torch.zeros(padded, width, dtype=torch.float16)
    tiles[:atoms] = value
    tiles = tiles.view(padded // 32, 32, width).transpose(1, 2).contiguous()
    d = torch.device("cuda:0")
    pitch = width + 8
    xd = torch.zeros(rows, pitch, dtype=dtype, device=d)
    xd[:, :width] = x.to(d)
    kd, vd = key_t.to(d), tiles.to(d)
    out = xd.view(out_dtype) if in_place else torch.full((rows + 1, pitch), float("nan"), dtype=out_dtype, device=d)
    beta_d = torch.tensor([abs(beta)], device=d).log()
    flags = (_lib.DA_ROUTE_UNIT_KEYS | (_lib.DA_ROUTE_NORMALIZE_INPUT if norm_in else 0)
             | (_lib.DA_ROUTE_NORMALIZE_OUTPUT if norm_out else 0) | (_lib.DA_ROUTE_BETA_IS_LOG if log_beta else 0))
    _lib.check(
        _lib.get().da_dictionary_route(
            xd.data_ptr(), rows, width, pitch, CODES[dtype], kd.data_ptr(), CODES[key_dtype], vd.data_ptr(), atoms,
            beta_d.data_ptr() if log_beta else None, _lib.DA_F32, 0.0 if log_beta else beta, 1e-6, flags, 1.0, 1.0,
            out.data_ptr(), pitch, CODES[out_dtype],
            torch.cuda.current_stream().cuda_stream,
        ),
        "route",
    )
    torch.cuda.synchronize()
    if not in_place:   # nothing is written past the rows or their width
        assert out[rows:].isnan().all() and out[:rows, width:].isnan().all()
    got = out[:rows, :width].double().cpu()

    u = x.double()
    if norm_in:
        u = u / u.norm(dim=-1, keepdim=True).clamp_min(1e-6)
    expected = torch.softmax(beta * (u @ key.double().t()), dim=-1) @ value.double()
    if norm_out:
        expected = expected / expected.norm(dim=-1, keepdim=True).clamp_min(1e-6)
    # The rounding of u moves a logit by eps/2 |u| |k| / sqrt(3) in all (the
    # coordinates' errors add as a random walk), its weight beta times that;
    # then one fp16 rounding of each weight and one of the output, and as much
    # again where normalization divides by a mean shorter than the atoms.
    eps = 2.0 ** (-8 if key_dtype == torch.bfloat16 else -11)
    out_eps = 2.0 ** (-8 if out_dtype == torch.bfloat16 else -11)
    bar = 2 * abs(beta) * eps / 3 ** 0.5 * 0.5 + 2 * 2.0 ** -11 + out_eps
    rel = ((got - expected).norm() / expected.norm()).item()
    assert got.isfinite().all() and rel <= bar, (rel, bar)


@pytest.mark.parametrize("beta", [8.0, 20.0])   # the fixed reference, row maxima
def test_route_tile_log_beta_on_the_device(beta) -> None:
    test_route_tile((200, 256, 130, torch.bfloat16, torch.float16, beta, True, True), False, log_beta=True)


@pytest.mark.parametrize("width", [256, 512])
@pytest.mark.parametrize("beta", [8.0, 30.0])
def test_route_tile_nan_rows(width, beta) -> None:
    """A NaN row is NaN in the output, and no other row sees it."""

    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    print(f"[route tile nan] {width} beta {beta}", flush=True)
    rows, atoms = 100, 200
    g = torch.Generator().manual_seed(7)
    d = torch.device("cuda:0")
    x = torch.randn(rows, width, generator=g).bfloat16().to(d)
    unit = F.normalize(torch.randn(256, width, generator=g), dim=-1).half()
    unit[atoms:] = 0
    kd = unit.to(d)
    vd = unit.view(8, 32, width).transpose(1, 2).contiguous().to(d)

    def route(x):
        out = torch.empty(rows, width, dtype=torch.float16, device=d)
        flags = _lib.DA_ROUTE_UNIT_KEYS | _lib.DA_ROUTE_NORMALIZE_INPUT | _lib.DA_ROUTE_NORMALIZE_OUTPUT
        _lib.check(
            _lib.get().da_dictionary_route(
                x.data_ptr(), rows, width, width, _lib.DA_BF16, kd.data_ptr(), _lib.DA_F16, vd.data_ptr(), atoms,
                None, _lib.DA_F32, beta, 1e-6, flags, 1.0, 1.0, out.data_ptr(), width, _lib.DA_F16,
                torch.cuda.current_stream().cuda_stream,
            ),
            "route",
        )
        torch.cuda.synchronize()
        return out.cpu()

    clean = route(x)
    spoilt = x.clone()
    spoilt[[3, 40, 99], 5] = float("nan")
    got = route(spoilt)
    bad = torch.zeros(rows, dtype=torch.bool)
    bad[[3, 40, 99]] = True
    assert got[bad].isnan().all() and clean.isfinite().all()
    assert torch.equal(got[~bad], clean[~bad])
