"""The small-tile ring GEMM (`gemm_ring_kernel`, tiles 18 to 26): every epilogue at the edges of its
tiles, of its ring and of its K loop. Its sums run in the order of the four-wave kernel on the same
MFMA, so every comparison is exact: against the 256 x 256 or 128 x 160 four-wave tile, which the
other tests compare with FP32 references."""

import pytest
import torch

from iris_mi355x import _lib
from iris_mi355x import kernels as K

pytestmark = pytest.mark.gpu
DEV = "cuda"
# tile -> (rows, columns, K tiles in the ring)
RING = {18: (32, 64, 8), 19: (64, 64, 8), 20: (96, 64, 7), 21: (128, 64, 6), 22: (32, 128, 7), 23: (64, 128, 6),
        24: (96, 128, 5), 25: (128, 128, 4), 26: (192, 128, 3)}


def forced(tile, fn):
    _lib.call("iris_gemm_force_tile", tile)
    try:
        return fn()
    finally:
        _lib.call("iris_gemm_force_tile", -1)


def randn(g, *shape, scale=1.0):
    return (scale * torch.randn(*shape, generator=g, device=DEV)).to(torch.bfloat16)


@pytest.mark.parametrize("tile", RING)
@pytest.mark.parametrize("extra_k", [0, 1, 2, 5])
@pytest.mark.parametrize("rows,cols", [(0, 1), (1, 0), (-1, -1), (None, None)])
def test_ring_tile_edges(tile, extra_k, rows, cols):
    """One row or column unit past or short of whole tiles, a single row, K loops of exactly the ring
    and of an odd and even number of tiles more; BF16 and FP32 output, bias, padded row strides."""
    bm, bn, stages = RING[tile]
    m = 1 if rows is None else 2 * bm + rows
    n = 4 if cols is None else 2 * bn + 4 * cols
    k = 64 * (stages + extra_k)
    g = torch.Generator(device=DEV).manual_seed(40 + extra_k)
    x, w = randn(g, m, k + 8)[:, :k], randn(g, n, k, scale=0.05)
    bias = torch.randn(n, generator=g, device=DEV)
    for kwargs in ({}, {"out_dtype": torch.float32}):
        for b in (None, bias):
            got = forced(tile, lambda: K.linear(x, w, b, **kwargs))
            want = forced(15, lambda: K.linear(x, w, b, **kwargs))
            assert torch.equal(got, want)
    prod = x.float().cpu() @ w.float().cpu().T  # k <= 832 products of N(0, 0.05): FP32 sums within 1e-4
    torch.testing.assert_close(forced(tile, lambda: K.linear(x, w, out_dtype=torch.float32)).cpu(), prod, rtol=1e-4,
                               atol=1e-4)


@pytest.mark.parametrize("tile", [t for t, (_, bn, _) in RING.items() if bn == 128])
@pytest.mark.parametrize("m,n", [(1, 64), (97, 320), (333, 448)])
def test_ring_swiglu(tile, m, n):
    g = torch.Generator(device=DEV).manual_seed(41)
    x, w = randn(g, m, 576), randn(g, n, 576, scale=0.05)
    for dtype in (torch.bfloat16, torch.float32):
        got = forced(tile, lambda: K.linear(x, w, swiglu=True, out_dtype=dtype))
        assert torch.equal(got, forced(16, lambda: K.linear(x, w, swiglu=True, out_dtype=dtype)))


@pytest.mark.parametrize("tile", [18, 20, 25])
@pytest.mark.parametrize("rows", [(60, 154), (1, 1), (64, 0)])
def test_ring_two_groups(tile, rows):
    g = torch.Generator(device=DEV).manual_seed(42)
    xs, ws = [randn(g, r, 640) for r in rows], [randn(g, 260, 640, scale=0.05) for _ in rows]
    outs = [[torch.empty(r, 260, device=DEV, dtype=torch.bfloat16) for r in rows] for _ in range(2)]
    forced(tile, lambda: K.linear_grouped(xs, ws, None, outs[0]))
    forced(16, lambda: K.linear_grouped(xs, ws, None, outs[1]))
    for got, want in zip(*outs):
        assert torch.equal(got, want)


@pytest.mark.parametrize("tile", [t for t, (_, bn, _) in RING.items() if bn == 128])
@pytest.mark.parametrize("heads,kv_heads,tokens,batch,gate", [(3, 1, (37,), 2, True), (2, 2, (60, 77), 1, False), (2, 1, (48, 80), 2, True),
                                                             (4, 2, (256,), 2, True), (2, 1, (256, 256), 1, True)])
def test_ring_qk_store(tile, heads, kv_heads, tokens, batch, gate):
    """The q | k | v (| gate) store on ring tiles writes what the plain product followed by
    qkv_prepare writes and nothing else: whole and ragged batch items and offsets, two streams, the V
    heads plain or transposed."""
    g = torch.Generator(device=DEV).manual_seed(43)
    n_qkv = (heads + 2 * kv_heads) * 128
    n = n_qkv + (128 * heads if gate else 0)
    v_col, k = (heads + kv_heads) * 128, 512
    offsets = [tokens[1], 0] if len(tokens) == 2 else [0]
    n_pad = (sum(tokens) + 63) // 64 * 64 + 64
    cos, sin = (torch.randn(n_pad, 64, generator=g, device=DEV) for _ in range(2))
    xs, ws = [randn(g, batch * t, k) for t in tokens], [randn(g, n, k, scale=0.05) for _ in tokens]
    gains = [[1 + 0.1 * torch.randn(128, generator=g, device=DEV) for _ in tokens] for _ in range(2)]

    def buffers():
        return [torch.full((batch, h, *s), 3.0, device=DEV, dtype=torch.bfloat16)
                for h, s in ((heads, (n_pad, 128)), (kv_heads, (n_pad, 128)), (kv_heads, (128, n_pad)))]

    q_ref, k_ref, vt_ref = buffers()
    plain = [forced(16, lambda x=x, w=w: K.linear(x, w)) for x, w in zip(xs, ws)]
    for out, qw, kw, t, off in zip(plain, *gains, tokens, offsets):
        K.qkv_prepare(out.view(batch, t, n), qw, kw, cos, sin, 1e-6, heads, kv_heads, q_ref, k_ref, vt_ref, 0,
                      heads * 128, v_col, off)
    for with_vt in (False, True):
        q, key, vt = buffers()
        outs = [torch.full((batch * t, n), 5.0, device=DEV, dtype=torch.bfloat16) for t in tokens]
        forced(tile, lambda: K.linear_qk_rope(xs, ws, outs, *gains, cos, sin, 1e-6, heads, kv_heads, q, key,
                                              list(tokens), offsets, vt=vt if with_vt else None, any_rows=True))
        assert torch.equal(q, q_ref) and torch.equal(key, k_ref)
        assert torch.equal(vt, vt_ref) if with_vt else torch.all(vt == 3.0)
        first = n_qkv if with_vt else v_col
        for out, ref in zip(outs, plain):
            assert torch.equal(out[:, first:], ref[:, first:]) and torch.all(out[:, :first] == 5.0)


@pytest.mark.parametrize("tokens,batch", [((300, 77), 1), ((272,), 2), ((256, 512), 1)])
def test_qkv_of_any_rows_without_ring_tiles(tokens, batch):
    """On the 256 x 256 store ragged items reach the V^T layout through the output's V columns."""
    g = torch.Generator(device=DEV).manual_seed(45)
    heads, kv_heads, k = 2, 1, 256
    n, v_col = 6 * 128, 3 * 128
    offsets = [tokens[1], 0] if len(tokens) == 2 else [0]
    n_pad = (sum(tokens) + 63) // 64 * 64
    cos, sin = (torch.randn(n_pad, 64, generator=g, device=DEV) for _ in range(2))
    xs, ws = [randn(g, batch * t, k) for t in tokens], [randn(g, n, k, scale=0.05) for _ in tokens]
    gains = [[torch.ones(128, device=DEV) for _ in tokens] for _ in range(2)]
    bufs = [[torch.full((batch, h, *s), 3.0, device=DEV, dtype=torch.bfloat16)
             for h, s in ((heads, (n_pad, 128)), (kv_heads, (n_pad, 128)), (kv_heads, (128, n_pad)))] for _ in range(2)]
    outs = [torch.empty(batch * t, n, device=DEV, dtype=torch.bfloat16) for t in tokens]
    for x, w, qw, kw, t, off in zip(xs, ws, *gains, tokens, offsets):
        plain = forced(16, lambda x=x, w=w: K.linear(x, w))
        K.qkv_prepare(plain.view(batch, t, n), qw, kw, cos, sin, 1e-6, heads, kv_heads, *bufs[0], 0, heads * 128, v_col,
                      off)
    forced(16, lambda: K.linear_qk_rope(xs, ws, outs, *gains, cos, sin, 1e-6, heads, kv_heads, *bufs[1][:2],
                                        list(tokens), offsets, vt=bufs[1][2], any_rows=True))
    for got, want in zip(bufs[1], bufs[0]):
        assert torch.equal(got, want)


def test_qk_store_of_whole_items_beside_an_empty_ragged_group():
    """Without rows a group's batch items do not matter: the 256 x 256 store still writes V^T itself and
    leaves the V columns of the output alone."""
    g = torch.Generator(device=DEV).manual_seed(48)
    k, n = 256, 6 * 128
    x, w = randn(g, 256, k), randn(g, n, k, scale=0.05)
    gain, cos, sin = torch.ones(128, device=DEV), *(torch.randn(256, 64, generator=g, device=DEV) for _ in range(2))
    plain = forced(16, lambda: K.linear(x, w))
    bufs = [[torch.full((1, h, *s), 3.0, device=DEV, dtype=torch.bfloat16)
             for h, s in ((2, (256, 128)), (1, (256, 128)), (1, (128, 256)))] for _ in range(2)]
    K.qkv_prepare(plain.view(1, 256, n), gain, gain, cos, sin, 1e-6, 2, 1, *bufs[0], 0, 256, 384)
    out = torch.full((256, n), 5.0, device=DEV, dtype=torch.bfloat16)
    P, q, key, vt = _lib.pointer_array, *bufs[1]
    twice = [P([t.data_ptr()] * 2) for t in (x, w, out, gain)]
    forced(16, lambda: _lib.call(
        "iris_gemm_bf16_qk_rope", 2, *twice[:3], _lib.int_array([256, 0]), n, k, k, k, n, twice[3], twice[3],
        _lib.int_array([256, 77]), _lib.int_array([0, 0]), cos.data_ptr(), sin.data_ptr(), 256, q.data_ptr(),
        key.data_ptr(), 2, 1, 256, vt.data_ptr(), 256, 1e-6, _lib.stream()))
    for got, want in zip(bufs[1], bufs[0]):
        assert torch.equal(got, want)
    assert torch.all(out[:, :512] == 5.0) and torch.equal(out[:, 512:], plain[:, 512:])


@pytest.mark.parametrize("tokens,batch", [((4096, 300), 1), ((1500,), 2), ((2000, 77), 1)])
def test_paired_qkv_store_of_ragged_items(tokens, batch):
    """q | k | v | gate of 20 query and 5 K/V heads at ragged row counts that the automatic choice runs
    as the 256 x 256 store paired with 288 x 160 gate columns (on 256 CUs), the V heads through the
    output: exactly the plain product and qkv_prepare."""
    g = torch.Generator(device=DEV).manual_seed(46)
    heads, kv_heads, k = 20, 5, 2560
    n, v_col, n_qkv = 50 * 128, 25 * 128, 30 * 128
    offsets = [tokens[1], 0] if len(tokens) == 2 else [0]
    n_pad = (sum(tokens) + 63) // 64 * 64
    cos, sin = (torch.randn(n_pad, 64, generator=g, device=DEV) for _ in range(2))
    xs, ws = [randn(g, batch * t, k) for t in tokens], [randn(g, n, k, scale=0.02) for _ in tokens]
    gains = [[1 + 0.1 * torch.randn(128, generator=g, device=DEV) for _ in tokens] for _ in range(2)]
    bufs = [[torch.full((batch, h, *s), 3.0, device=DEV, dtype=torch.bfloat16)
             for h, s in ((heads, (n_pad, 128)), (kv_heads, (n_pad, 128)), (kv_heads, (128, n_pad)))] for _ in range(2)]
    plain = [forced(15, lambda x=x, w=w: K.linear(x, w)) for x, w in zip(xs, ws)]
    for out, qw, kw, t, off in zip(plain, *gains, tokens, offsets):
        K.qkv_prepare(out.view(batch, t, n), qw, kw, cos, sin, 1e-6, heads, kv_heads, *bufs[0], 0, heads * 128, v_col,
                      off)
    outs = [torch.full((batch * t, n), 5.0, device=DEV, dtype=torch.bfloat16) for t in tokens]
    K.linear_qk_rope(xs, ws, outs, *gains, cos, sin, 1e-6, heads, kv_heads, *bufs[1][:2], list(tokens), offsets,
                     vt=bufs[1][2], any_rows=True)
    for got, want in zip(bufs[1], bufs[0]):
        assert torch.equal(got, want)
    for out, ref in zip(outs, plain):
        assert torch.equal(out[:, n_qkv:], ref[:, n_qkv:]) and torch.all(out[:, :v_col] == 5.0)


def test_ring_refuses_a_k_loop_shorter_than_its_ring():
    x, w = torch.zeros(8, 128, device=DEV, dtype=torch.bfloat16), torch.zeros(64, 128, device=DEV, dtype=torch.bfloat16)
    with pytest.raises(Exception, match="ring"):
        forced(19, lambda: K.linear(x, w))
    assert torch.all(K.linear(x, w) == 0)  # the automatic choice takes another tile


@pytest.mark.parametrize("k", [64, 128, 192])
@pytest.mark.parametrize("m", [1, 77, 333])
def test_automatic_choice_for_k_loops_around_the_smallest_ring(k, m):
    """One and two K tiles fit no ring, three the smallest one only."""
    g = torch.Generator(device=DEV).manual_seed(47)
    x, w = randn(g, m, k), randn(g, 448, k, scale=0.1)
    for kwargs in ({}, {"out_dtype": torch.float32}, {"swiglu": True}):
        assert torch.equal(K.linear(x, w, **kwargs), forced(16, lambda: K.linear(x, w, **kwargs)))
    prod = x.double() @ w.double().T  # k <= 192 products of N(0, 0.1): FP32 sums within 1e-5
    torch.testing.assert_close(K.linear(x, w, out_dtype=torch.float32).double(), prod, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("n,k,swiglu", [(2560, 2560, False), (13696, 2560, True), (2560, 6848, False)])
def test_automatic_choice_over_row_counts_is_row_independent(n, k, swiglu):
    """A row's result does not depend on how many rows the call has, so on which tile runs it."""
    g = torch.Generator(device=DEV).manual_seed(44)
    x, w = randn(g, 1500, k), randn(g, n, k, scale=0.02)
    whole = K.linear(x, w, swiglu=swiglu)
    for m in (1, 40, 130, 333, 520, 900):
        assert torch.equal(K.linear(x[:m], w, swiglu=swiglu), whole[:m])


@pytest.mark.parametrize("m,n,k,swiglu", [(1280, 3840, 512, False), (1153, 4096, 1280, False), (4097, 4096, 1280, False),
                                          (3586, 13696, 2560, True), (5000, 13696, 2560, True), (3590, 5504, 1280, True)])
def test_automatic_plans_are_the_four_wave_tile_bit_for_bit(m, n, k, swiglu):
    """On either side of the plan rules: one round of ring or four-wave tiles, columns left over after whole
    rounds on ring tiles or in a pair."""
    g = torch.Generator(device=DEV).manual_seed(49)
    x, w = randn(g, m, k), randn(g, n, k, scale=0.02)
    assert torch.equal(K.linear(x, w, swiglu=swiglu), forced(16, lambda: K.linear(x, w, swiglu=swiglu)))
