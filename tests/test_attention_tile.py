"""The eight-wave attention kernel.

Calls the C entry point at the sizes where the tiling can go wrong (edges of
the 128-query and 32-key tiles, split and whole key ranges, one and two
value slices), against the NumPy oracle.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from double_attention import _lib

pytestmark = pytest.mark.gpu

F16, BF16 = _lib.DA_F16, _lib.DA_BF16


def _case(batch, maps, length, score_dim, value_dim, dtype, causal, log_scale, bound, out_f32=False, spoil=None,
          pad=0):
    g = torch.Generator().manual_seed(length + score_dim)
    rows = torch.nn.functional.normalize(torch.randn(batch, length, 2, maps, score_dim, generator=g), dim=-1).half()
    value = torch.randn(batch, length, value_dim, generator=g).to(dtype)
    if spoil is not None:
        spoil(rows, value)
    scales = torch.linspace(log_scale - 0.4, log_scale + 0.4, maps) if maps > 1 else torch.tensor([log_scale])
    logits = torch.linspace(-0.7, 0.9, maps)
    padded = (length + 63) // 64 * 64
    tiles = torch.zeros(batch, padded // 32, value_dim, 32, dtype=dtype)
    full = torch.zeros(batch, padded, value_dim, dtype=dtype)
    full[:, :length] = value
    tiles.copy_(full.view(batch, padded // 32, 32, value_dim).transpose(2, 3))

    d = torch.device("cuda:0")
    rd, td, sd, ld = rows.to(d), tiles.to(d), scales.to(d), logits.to(d)
    out_dtype = torch.float32 if out_f32 else dtype
    # `pad` features before the output's first and after each row's last.
    whole = torch.full((pad + batch * length * (value_dim + pad),), float("nan"), dtype=out_dtype, device=d)
    framed = whole[pad:].view(batch, length, value_dim + pad)
    out = framed[..., :value_dim]
    flags = _lib.DA_ATTN_SCALES_ARE_LOG | (_lib.DA_ATTN_CAUSAL if causal else 0)
    flags |= (_lib.DA_ATTN_MIX if maps > 1 else 0) | (_lib.DA_ATTN_OUT_F32 if out_f32 else 0)
    lib = _lib.get()
    need = lib.da_attention_workspace_bytes(batch, maps, length, score_dim, value_dim, flags)
    workspace = torch.empty(max(need, 1), dtype=torch.uint8, device=d)
    width = maps * score_dim

    def call(nbytes):
        whole.fill_(float("nan"))
        _lib.check(
            lib.da_routed_attention(
                rd.data_ptr(), rd.data_ptr() + width * 2, length * 2 * width, 2 * width, score_dim, 1, score_dim,
                td.data_ptr(), td.stride(0), batch, maps, length, value_dim, sd.data_ptr(), _lib.DA_F32, 1.0,
                ld.data_ptr() if maps > 1 else None, _lib.DA_F32, flags, bound,
                F16, BF16 if dtype == torch.bfloat16 else F16, out.data_ptr(), out.stride(0), out.stride(1), 0,
                workspace.data_ptr() if nbytes else None, nbytes, torch.cuda.current_stream().cuda_stream,
            ),
            "attention",
        )
        torch.cuda.synchronize()
        assert whole[:pad].isnan().all() and framed[..., value_dim:].isnan().all()
        return out.float().cpu().numpy()

    q, k = (rows[:, :, i].permute(0, 2, 1, 3).float().numpy() for i in (0, 1))
    per_map = oracle.routed_attention(q, k, value.float().numpy(), np.exp(scales.numpy()), causal)
    alpha = torch.softmax(logits, 0).numpy() if maps > 1 else np.ones(1, np.float32)
    return call, need, np.einsum("s,bstd->btd", alpha, per_map)


@pytest.mark.parametrize("case", [
    # batch, maps, length, score width, value width, dtype, causal, log scale, bound, fp32 out
    (1, 1, 2048, 256, 512, torch.bfloat16, True, 2.77, 1.01, False),
    (1, 1, 2081, 256, 512, torch.bfloat16, True, 2.77, 1.01, True),      # ragged last tiles, fp32 pieces
    (1, 1, 2111, 256, 768, torch.float16, True, 2.77, 1.01, False),      # row maxima first, three 256-wide slices
    (1, 1, 2049, 256, 256, torch.bfloat16, False, 6.0, 1.01, False),     # scale past the fixed reference
    (1, 1, 2177, 256, 512, torch.bfloat16, False, 2.77, 1.01, False),    # split without a mask
    (1, 1, 1024, 512, 512, torch.bfloat16, True, 3.1, 1.01, False),
    (2, 1, 1055, 512, 256, torch.float16, True, 3.1, 0.0, True),         # no bound
    (9, 1, 1024, 512, 256, torch.bfloat16, False, 3.1, 1.01, False),     # whole key ranges
])
def test_attention_tile(case) -> None:
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    print(f"[attention tile] {case}", flush=True)
    call, need, expected = _case(*case)
    assert need > 0 or case[0] == 9
    got = call(need)
    # One 16-bit rounding of P, V and the output each, averaged over the keys:
    # well under the operand type's half unit in the last place.
    bar = 5e-3 if case[5] == torch.bfloat16 else 1e-3
    rel = np.linalg.norm(got - expected) / np.linalg.norm(expected)
    assert np.isfinite(got).all() and rel <= bar, rel
    # Without scratch the general kernel takes the call.
    general = call(0)
    assert np.linalg.norm(general - got) / np.linalg.norm(expected) <= 2 * bar


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])   # the fixed reference, and row maxima
@pytest.mark.parametrize(("length", "width", "causal"), [
    (2177, 256, True),
    (2177, 512, True),
    (2177, 256, False),
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

    args = (1, 1, length, width, 512, dtype, causal, 2.77, 1.01)
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
    args = (batch, 1, length, width, value_dim, dtype, causal, 2.77, 1.01)
    call, need, _ = _case(*args)
    exact, need32, _ = _case(*args, out_f32=True)
    assert need > 0 and need32 > 0   # both split
    rounded = torch.from_numpy(exact(need32)).to(dtype).float().numpy()
    np.testing.assert_array_equal(call(need), rounded)


@pytest.mark.parametrize("batch", [1, 24])   # split keys (the merge stores the output), whole ones
def test_attention_tile_eight_byte_outputs(batch) -> None:
    """16-bit outputs that start and step at multiples of 8 bytes, not of 16."""

    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    print(f"[attention tile 8-byte outputs] batch {batch}", flush=True)
    args = (batch, 1, 1055, 512, 256, torch.bfloat16, False, 3.1, 1.01)
    plain, need, _ = _case(*args)
    assert (need > 0) == (batch == 1)
    framed, _, _ = _case(*args, pad=4)
    np.testing.assert_array_equal(framed(need), plain(need))
