"""GPU parity of attention over several queries (prompts and prompt chunks)
against the oracle (src/core/TensorCalc.cpp:1167-1314): the MFMA prefill
kernel's row and key tile edges, windows, offsets past the keys, page lists,
and non-finite keys and values."""
import numpy as np
import pytest
import torch

from tests.helpers import assert_close, from_f32, normal, rng, to_oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from sandyrt_amd import ops
    return ops


def pages_of(ops, t, P, shift=0):
    """A [B, Hkv, T, D] tensor as a page list (its own allocation a page,
    `shift` elements into it) and the tensors to keep alive."""
    B, H, T, D = t.shape
    keep, at = [], []
    for p in range((T + P - 1) // P):
        page = torch.zeros(B * H * P * D + shift, dtype=t.dtype, device="cuda")
        rows = t[:, :, p * P:(p + 1) * P].reshape(B * H, -1, D)
        page[shift:].view(B * H, P, D)[:, :rows.shape[1]] = rows
        keep.append(page)
        at.append(page.data_ptr() + shift * t.element_size())
    return ops.PagedView(torch.tensor(at, dtype=torch.int64, device="cuda"), t.shape, P, t.dtype), keep


def check(ops, oracle, dtype, B, hq, hkv, tq, tk, D, pos, window, P=0, shift=0, spoil=None, heads_inner=False, kv_room=0):
    r = rng(tq * 131 + tk + D + window)
    q = from_f32(normal(r, (B, hq, tq, D), 0.5), dtype)
    if heads_inner:  # the engine's [B, T, H, D] rows seen as [B, H, T, D]
        q = q.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3)
    k = from_f32(normal(r, (B, hkv, tk, D), 0.5), dtype)
    v = from_f32(normal(r, (B, hkv, tk, D)), dtype)
    if spoil:
        spoil(k, v)
    if kv_room:  # views of [B, T + room, Hkv, D] caches: the heads inside the tokens, keys past the last
        k, v = (torch.cat([t, torch.full_like(t[:, :, :1], float("nan")).expand(-1, -1, kv_room, -1)], 2)
                .permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3)[:, :, :tk] for t in (k, v))
        assert not k.is_contiguous() and k.stride(2) == hkv * D
    p = torch.tensor(pos, device="cuda") if pos is not None else None
    want = oracle.attention(to_oracle(q.contiguous()), to_oracle(k), to_oracle(v),
                            np.array(pos, np.int64) if pos is not None else None, window, -1.0)
    out = torch.empty_like(q)
    if P:
        kv, keep_k = pages_of(ops, k, P, shift)
        vv, keep_v = pages_of(ops, v, P, shift)
        ops.attention_paged_view(q, kv, vv, p, window, out=out)
    else:
        ops.attention(q, k, v, p, window, out=out)
    ops.check_device_errors()
    what = f"B{B} hq{hq} hkv{hkv} tq{tq} tk{tk} D{D} pos{pos} w{window} P{P}"
    if dtype == torch.float32:
        # an output is a weighted mean of v: the reference's in-order sum and the
        # MFMA sums round partial sums of at most max |v| some dozen times to
        # 2^-24 of them, so elements near zero are held to 8 of those roundings
        got, want, big = to_oracle(out.contiguous()), np.asarray(want), float(np.abs(to_oracle(v)[np.isfinite(to_oracle(v))]).max())
        np.testing.assert_allclose(got, want, rtol=1e-5, atol=8 * 2.0 ** -24 * big, err_msg=what)
    else:
        assert_close(out.contiguous(), want, dtype, what)


SHAPES = [
    # one row tile and less, more keys than queries, several queries a tile column
    dict(B=1, hq=1, hkv=1, tq=2, tk=2, D=64, pos=None, window=0),
    dict(B=2, hq=8, hkv=2, tq=9, tk=40, D=64, pos=[31, 5], window=0),
    dict(B=1, hq=8, hkv=1, tq=37, tk=200, D=64, pos=[163], window=0),
    # several row tiles with a ragged end; a group that does not divide the tile
    dict(B=1, hq=6, hkv=2, tq=65, tk=65, D=64, pos=None, window=0),
    dict(B=1, hq=12, hkv=12, tq=130, tk=130, D=64, pos=[0], window=0),
    dict(B=1, hq=4, hkv=2, tq=67, tk=131, D=128, pos=[64], window=0),
    dict(B=2, hq=4, hkv=1, tq=33, tk=97, D=256, pos=[64, 3], window=0),
    # windows: inside a tile, across tiles; rows that see no key
    dict(B=1, hq=4, hkv=2, tq=50, tk=150, D=64, pos=[100], window=7),
    dict(B=1, hq=4, hkv=2, tq=50, tk=250, D=128, pos=[190], window=100),
    dict(B=2, hq=2, hkv=1, tq=40, tk=60, D=256, pos=[30, 200], window=33),
    # offsets past the last key
    dict(B=1, hq=2, hkv=2, tq=35, tk=70, D=64, pos=[500], window=0),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows", ["", "1", "2"])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_prefill_matches_oracle(ops, oracle, monkeypatch, shape, rows, dtype):
    """Every row-tile form (32 rows a workgroup with the keys split over four
    waves, 64 over two) and the one chosen by size."""
    if rows:
        monkeypatch.setenv("SANDY_PREFILL_RW", rows)
    check(ops, oracle, dtype, **shape)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", [SHAPES[2], SHAPES[5], SHAPES[9]], ids=str)
def test_prefill_strided_heads_and_pages(ops, oracle, shape, dtype):
    """q and out with the heads inside the tokens; K/V from page lists of 1,
    16 and 64 rows, also where pages start on odd elements."""
    check(ops, oracle, dtype, heads_inner=True, **shape)
    for P, shift in ((1, 0), (16, 0), (64, 8), (16, 3)):
        check(ops, oracle, dtype, P=P, shift=shift, **shape)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", [SHAPES[1], SHAPES[5], SHAPES[8]], ids=str)
def test_prefill_strided_keys_and_values(ops, oracle, monkeypatch, shape, dtype):
    """Dense K/V that are views of larger caches with the heads inside the
    tokens; what lies past the keys is never used.  The general kernel takes
    the same views."""
    check(ops, oracle, dtype, kv_room=5, **shape)
    monkeypatch.setenv("SANDY_PREFILL_GENERAL", "1")
    check(ops, oracle, dtype, kv_room=5, **shape)


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 64), (torch.bfloat16, 256), (torch.float32, 64)])
@pytest.mark.parametrize("rows", ["1", "2"])
@pytest.mark.parametrize("tk,window", [(511, 0), (512, 0), (700, 0), (700, 300), (700, 600)])
def test_prefill_long_page_lists(ops, oracle, monkeypatch, tk, window, rows, dtype, D):
    """Pages of one key: 512 page addresses, the most that are held in LDS, and
    more (read from memory per chunk), aligned ones too; a window that brings a
    longer list under the line and one that does not."""
    monkeypatch.setenv("SANDY_PREFILL_RW", rows)
    check(ops, oracle, dtype, B=1, hq=4, hkv=2, tq=40, tk=tk, D=D, pos=[tk - 40], window=window, P=1)


@pytest.mark.parametrize("rows", ["1", "2"])
@pytest.mark.parametrize("window", [200, 201, 5000, 2 ** 63 - 66, 2 ** 63 - 2, 2 ** 63 - 1])
def test_prefill_window_wider_than_the_keys_over_pages(ops, oracle, monkeypatch, window, rows):
    """Windows of all the keys and more, up to the largest value (no limit)."""
    monkeypatch.setenv("SANDY_PREFILL_RW", rows)
    check(ops, oracle, torch.bfloat16, B=1, hq=8, hkv=1, tq=37, tk=200, D=64, pos=[163], window=window, P=16)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("P", [0, 16])
def test_prefill_non_finite_values_reach_only_their_rows(ops, oracle, P, dtype):
    """An infinity or NaN in V, or a NaN in K, changes the rows that see its
    key and no other (the reference never reads a masked key)."""
    def spoil(k, v):
        v[0, 0, 70, 3] = float("inf")
        v[0, 1, 90, 5] = float("nan")
        v[0, 1, 20, 6] = float("-inf")
        k[0, 0, 95, 1] = float("nan")
        k[0, 1, 98, 2] = float("inf")
    check(ops, oracle, dtype, B=1, hq=4, hkv=2, tq=60, tk=100, D=64, pos=[40], window=30, P=P, spoil=spoil)


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 64), (torch.bfloat16, 128), (torch.bfloat16, 256),
                                     (torch.float32, 64), (torch.float32, 128)])
@pytest.mark.parametrize("rows", ["1", "2"])
@pytest.mark.parametrize("window,P,shift", [(0, 0, 0), (130, 16, 0), (0, 16, 3)])
def test_prefill_non_finite_values_over_several_key_chunks(ops, oracle, monkeypatch, window, P, shift, rows, dtype, D):
    """The rows computed again, in every form: infinities of both signs in one
    column, NaN, an infinite key (its score is NaN, an infinity or -inf) and a
    key of score -inf under an infinite value, at chunk edges."""
    def spoil(k, v):
        v[0, 0, 0, 3] = float("inf")
        v[0, 0, 127, 3] = float("-inf")
        v[0, 0, 128, D - 1] = float("nan")
        v[0, 1, 190, 5] = float("-inf")
        k[0, 1, 200, :] = float("-inf")
        v[0, 1, 200, 0] = float("inf")
        k[0, 1, 240, 2] = float("nan")
    monkeypatch.setenv("SANDY_PREFILL_RW", rows)
    check(ops, oracle, dtype, B=1, hq=6, hkv=2, tq=90, tk=260, D=D, pos=[165], window=window, P=P, shift=shift, spoil=spoil)


@pytest.mark.parametrize("scale", [1.0, 2.0 ** 14, 2.0 ** 20])
def test_prefill_large_scores(ops, oracle, scale):
    """Scores up to 2^40: past 2^31 the exponent's rounding alone leaves the range
    of exp2, and the rows are computed again in the general kernel's arithmetic."""
    r = rng(5)
    q, k = (from_f32(normal(r, (1, h, n, 64), scale), torch.bfloat16) for h, n in ((4, 40), (2, 150)))
    v = from_f32(normal(r, (1, 2, 150, 64)), torch.bfloat16)
    pos = torch.tensor([110], device="cuda")
    want = oracle.attention(to_oracle(q), to_oracle(k), to_oracle(v), np.array([110]), 0, -1.0)
    assert_close(ops.attention(q, k, v, pos), want, torch.bfloat16, f"scale {scale}")


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 64), (torch.bfloat16, 256), (torch.float32, 128)])
@pytest.mark.parametrize("rows", ["1", "2"])
def test_prefill_in_place(ops, oracle, monkeypatch, rows, dtype, D):
    """`out` may be `q`, also where rows are computed again for an infinity in V."""
    monkeypatch.setenv("SANDY_PREFILL_RW", rows)
    r = rng(D)
    for bad in (None, float("inf")):
        q, k = from_f32(normal(r, (1, 4, 70, D), 0.5), dtype), from_f32(normal(r, (1, 2, 90, D), 0.5), dtype)
        v = from_f32(normal(r, (1, 2, 90, D)), dtype)
        if bad is not None:
            v[0, 0, 50, 3] = bad
            v[0, 1, 2, 5] = bad
        pos = torch.tensor([20], device="cuda")
        want = ops.attention(q, k, v, pos)
        got = ops.attention(q, k, v, pos, out=q)
        assert got.data_ptr() == q.data_ptr() and torch.equal(got, want)
        assert torch.isfinite(got).all() == (bad is None)


def test_prefill_errors(ops):
    """A negative offset and a null page are recorded."""
    from sandyrt_amd._lib import SandyError
    q = torch.zeros(1, 2, 4, 64, dtype=torch.bfloat16, device="cuda")
    k = torch.zeros(1, 1, 20, 64, dtype=torch.bfloat16, device="cuda")
    ops.attention(q, k, k, torch.tensor([-1], device="cuda"))
    with pytest.raises(SandyError, match="attention position_offsets must be non-negative"):
        ops.check_device_errors()
    view, keep = pages_of(ops, k, 16)
    view.pages[1] = 0
    ops.attention_paged_view(q, view, view, torch.tensor([4], device="cuda"))  # keys 0..7: page 0 alone
    ops.check_device_errors()
    ops.attention_paged_view(q, view, view, torch.tensor([14], device="cuda"))
    with pytest.raises(SandyError, match="block id outside the pool"):
        ops.check_device_errors()


@pytest.mark.parametrize("dtype,D,tq,past,spread", [
    (torch.float32, 64, 2, 0, 1.0), (torch.float32, 128, 2, 0, 3.0), (torch.float32, 64, 64, 0, 1.0),
    (torch.float32, 128, 5, 300, 1.0), (torch.bfloat16, 64, 64, 0, 1.0), (torch.bfloat16, 128, 40, 200, 1.0),
    (torch.bfloat16, 256, 33, 100, 1.0)])
def test_prefill_error_against_64_bits(ops, monkeypatch, dtype, D, tq, past, spread):
    """No further from the exact outputs than the general kernel, over enough
    rows for the difference to show: the 2-norm of the error in f32, in bf16
    the share of outputs that are not the nearest value to the exact one."""
    g = torch.Generator(device="cuda").manual_seed(D + tq + past)
    B, tk = max(4, min(512, 6000 // (tq + past))), tq + past
    q, k, v = (torch.randn(B, 12, n, D, generator=g, device="cuda") for n in (tq, tk, tk))
    q, k, v = (q * spread).to(dtype), k.to(dtype), v.to(dtype)
    pos = torch.full((B,), past, dtype=torch.int64, device="cuda")
    s = q.double() @ k.double().transpose(2, 3).contiguous() / D ** 0.5
    seen = torch.arange(tk, device="cuda") <= past + torch.arange(tq, device="cuda")[:, None]
    want = torch.softmax(s.masked_fill(~seen, float("-inf")), -1) @ v.double()

    def error():
        out = ops.attention(q, k, v, pos)
        if dtype == torch.float32:
            return ((out.double() - want).norm() / want.norm()).item()
        return (out != want.to(dtype)).double().mean().item()

    here = error()
    monkeypatch.setenv("SANDY_PREFILL_GENERAL", "1")
    general = error()
    assert here <= general, f"{here:.4e} against {general:.4e}"
