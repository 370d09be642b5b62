"""The eight-wave attention kernel.

Calls the C entry point at the sizes where the tiling can go wrong (edges of
the 128-query and 32-key tiles, split and whole key ranges, one to three
value slices), against the NumPy oracle.  The shapes are ones that the rule
between the two attention kernels gives to this one.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from double_attention import _lib

pytestmark = pytest.mark.gpu

F16, BF16 = _lib.DA_F16, _lib.DA_BF16


def _case(batch, length, score_dim, value_dim, dtype, causal, log_scale, bound, out_f32=False, spoil=None, pad=0):
    """A function that runs the call with so many bytes of scratch, the scratch
    it can use, and the oracle's output."""

    g = torch.Generator().manual_seed(length + score_dim)
    rows = torch.nn.functional.normalize(torch.randn(batch, length, 2, score_dim, generator=g), dim=-1).half()
    value = torch.randn(batch, length, value_dim, generator=g).to(dtype)
    if spoil is not None:
        spoil(rows, value)
    pitch = 2 * score_dim + 8   # q and k side by side, and a gap
    pitched = torch.zeros(batch, length, pitch, dtype=torch.float16)
    pitched[..., :2 * score_dim] = rows.flatten(2)
    padded = (length + 63) // 64 * 64
    tiles = torch.zeros(batch, padded // 32, value_dim, 32, dtype=dtype)
    full = torch.zeros(batch, padded, value_dim, dtype=dtype)
    full[:, :length] = value
    tiles.copy_(full.view(batch, padded // 32, 32, value_dim).transpose(2, 3))

    d = torch.device("cuda:0")
    rd, td, sd = pitched.to(d), tiles.to(d), torch.tensor([log_scale], device=d)
    out_dtype = torch.float32 if out_f32 else dtype
    # `pad` features before the output's first and after each row's last.
    whole = torch.full((pad + batch * length * (value_dim + pad),), float("nan"), dtype=out_dtype, device=d)
    framed = whole[pad:].view(batch, length, value_dim + pad)
    out = framed[..., :value_dim]
    flags = _lib.DA_ATTN_SCALES_ARE_LOG | (_lib.DA_ATTN_CAUSAL if causal else 0)
    flags |= _lib.DA_ATTN_OUT_F32 if out_f32 else 0
    lib = _lib.get()
    need = lib.da_attention_workspace_bytes(batch, 1, length, score_dim, value_dim, flags)
    workspace = torch.empty(max(need, 1), dtype=torch.uint8, device=d)

    def call(nbytes):
        whole.fill_(float("nan"))
        _lib.check(
            lib.da_routed_attention(
                rd.data_ptr(), rd.data_ptr() + score_dim * 2, length * pitch, pitch, score_dim, 1, score_dim,
                td.data_ptr(), td.stride(0), batch, 1, length, value_dim, sd.data_ptr(), _lib.DA_F32, 1.0,
                None, _lib.DA_F32, flags, bound,
                F16, BF16 if dtype == torch.bfloat16 else F16, out.data_ptr(), out.stride(0), out.stride(1), 0,
                workspace.data_ptr() if nbytes else None, nbytes, torch.cuda.current_stream().cuda_stream,
            ),
            "attention",
        )
        torch.cuda.synchronize()
        assert whole[:pad].isnan().all() and framed[..., value_dim:].isnan().all()
        return out.float().cpu().numpy()

    q, k = (rows[:, None, :, i].float().numpy() for i in (0, 1))
    scales = np.exp(np.array([log_scale], np.float32))
    return call, need, oracle.routed_attention(q, k, value.float().numpy(), scales, causal)[:, 0]


def _close(got, expected, dtype) -> None:
    # One 16-bit rounding of P, V and the output each, averaged over the keys:
    # well under the operand type's half unit in the last place.
    bar = 5e-3 if dtype == torch.bfloat16 else 1e-3
    rel = np.linalg.norm(got - expected) / np.linalg.norm(expected)
    assert np.isfinite(got).all() and rel <= bar, rel


@pytest.mark.parametrize("case", [
    # batch, length, score width, value width, dtype, causal, log scale, bound, fp32 out
    (1, 2048, 256, 512, torch.bfloat16, True, 2.77, 1.01, False),
    (1, 2081, 256, 512, torch.bfloat16, True, 2.77, 1.01, True),      # ragged last tiles, fp32 pieces
    (1, 4127, 256, 768, torch.float16, True, 2.77, 1.01, False),      # row maxima first, three 256-wide slices
    (1, 2561, 256, 512, torch.bfloat16, False, 6.0, 1.01, False),     # scale past the fixed reference
    (1, 2433, 256, 512, torch.bfloat16, False, 2.77, 1.01, False),    # split without a mask
    (1, 1024, 512, 512, torch.bfloat16, True, 3.1, 1.01, False),
    (2, 1055, 512, 256, torch.bfloat16, True, 3.1, 0.0, True),        # no bound
    (9, 1100, 512, 256, torch.bfloat16, False, 3.1, 1.01, False),     # two pieces
])
def test_attention_tile(case) -> None:
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    print(f"[attention tile] {case}", flush=True)
    call, need, expected = _case(*case)
    assert need > 0
    got = call(need)
    _close(got, expected, case[4])
    # Without scratch the general kernel takes the call.
    general = call(0)
    _close(general, expected, case[4])
    assert (general != got).any()


@pytest.mark.parametrize("case", [
    (11, 2048, 256, 512, torch.bfloat16, False, 2.77, 1.01, False),
    (24, 1100, 512, 256, torch.bfloat16, False, 3.1, 1.01, False),
    (40, 1055, 512, 256, torch.bfloat16, True, 3.1, 1.01, True),
])
def test_attention_tile_whole_key_ranges(case) -> None:
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    print(f"[attention tile whole] {case}", flush=True)
    call, need, expected = _case(*case)
    assert need == 0
    _close(call(0), expected, case[4])


def test_attention_tile_with_less_scratch() -> None:
    """Less scratch than this kernel can use, but enough for the general
    kernel's split: the call is taken, by that one."""

    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    print("[attention tile less scratch]", flush=True)
    call, need, expected = _case(1, 4096, 256, 512, torch.bfloat16, True, 2.77, 1.01)
    full = call(need)
    less = call(need - 256)
    _close(full, expected, torch.bfloat16)
    _close(less, expected, torch.bfloat16)
    assert (full != less).any()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])   # the fixed reference, and row maxima
@pytest.mark.parametrize(("length", "width", "causal"), [
    (4097, 256, True),
    (2177, 512, True),    # fp16: the general kernel
    (2500, 256, False),
    (1500, 256, True),    # the general kernel
    (1500, 256, False),
])
def test_split_attention_nan_scores(dtype, length, width, causal) -> None:
    """A NaN key reaches every query that sees it, a NaN query its own row, in
    split and whole query tiles alike; no other row changes."""

    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    print(f"[split attention nan] {dtype} {length} {width} causal {causal}", flush=True)
    key_at, query_at = 1400, (5, 700, 1300)

    def spoil(rows, value):
        rows[0, key_at, 1] = float("nan")
        for t in query_at:
            rows[0, t, 0] = float("nan")

    args = (1, length, width, 512, dtype, causal, 2.77, 1.01)
    call, need, _ = _case(*args)
    clean = call(need)[0]
    call, need, _ = _case(*args, spoil=spoil)
    assert need > 0
    got = call(need)[0]
    bad = np.zeros(length, bool)
    bad[key_at if causal else 0:] = True
    bad[list(query_at)] = True
    assert np.isnan(got[bad]).all(), np.flatnonzero(bad & ~np.isnan(got).all(axis=1))[:8]
    np.testing.assert_array_equal(got[~bad], clean[~bad])


@pytest.mark.parametrize("case", [
    # batch, length, score width, value width, causal: the general kernel splits none of these
    (2, 2500, 256, 512, False),
    (3, 2500, 256, 512, True),
    (4, 2048, 512, 512, False),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_attention_tile_pieces_are_fp32(case, dtype) -> None:
    """Where only this kernel splits the keys, a 16-bit output is its fp32 one
    rounded once: the pieces hold fp32."""

    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    batch, length, width, value_dim, causal = case
    print(f"[attention tile pieces] {case} {dtype}", flush=True)
    args = (batch, length, width, value_dim, dtype, causal, 2.77, 1.01)
    call, need, _ = _case(*args)
    exact, need32, _ = _case(*args, out_f32=True)
    assert need > 0 and need32 > 0   # both split
    rounded = torch.from_numpy(exact(need32)).to(dtype).float().numpy()
    np.testing.assert_array_equal(call(need), rounded)


@pytest.mark.parametrize(("batch", "length"), [(1, 1100), (24, 1100)])   # split keys (the merge stores the output), whole
def test_attention_tile_eight_byte_outputs(batch, length) -> None:
    """16-bit outputs that start and step at multiples of 8 bytes, not of 16."""

    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    print(f"[attention tile 8-byte outputs] batch {batch}", flush=True)
    args = (batch, length, 512, 256, torch.bfloat16, False, 3.1, 1.01)
    plain, need, _ = _case(*args)
    assert (need > 0) == (batch == 1)
    framed, _, _ = _case(*args, pad=4)
    np.testing.assert_array_equal(framed(need), plain(need))
