"""The row kernels with a workgroup per row: widths at the edges of their chunk layout (8 columns per
thread, 512 per wave), single rows and two streams, against FP64; and the two forms of
``rms_norm_modulate`` and the gated residual (chosen by row count and input dtype), which agree bit
for bit."""

import pytest
import torch

from iris_mi355x import kernels as K

pytestmark = pytest.mark.gpu
DEV = "cuda"
WIDTHS = [128, 384, 512, 640, 1024, 1664, 2560, 2688, 4096, 8192]


def norm64(x, w):
    x = x.double()
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * w.double()


@pytest.mark.parametrize("width", WIDTHS)
@pytest.mark.parametrize("dtype,rows", [(torch.float32, 1600), (torch.bfloat16, 600)])
def test_rms_norm_modulate_forms_agree(width, dtype, rows):
    g = torch.Generator(device=DEV).manual_seed(70)
    x = torch.randn(1, rows, width, generator=g, device=DEV).to(dtype)
    w = 1 + 0.1 * torch.randn(width, generator=g, device=DEV)
    shift, scale = (0.1 * torch.randn(1, 1, width, generator=g, device=DEV) for _ in range(2))
    whole = K.rms_norm_modulate(x, w, shift, scale, 1e-6, torch.float32)
    for n in (1, 3, 64, 333):
        part = K.rms_norm_modulate(x[:, :n].contiguous(), w, shift, scale, 1e-6, torch.float32)
        assert torch.equal(part, whole[:, :n])
    want = norm64(x, w) * (1 + scale.double()) + shift.double()
    # FP32 sums over at most 8192 squares and a few roundings of values below ~6
    torch.testing.assert_close(whole.double(), want, rtol=2e-6, atol=4e-6)


@pytest.mark.parametrize("width", WIDTHS)
@pytest.mark.parametrize("rows", [(1, 1), (5, 77)])
@pytest.mark.parametrize("branch_dtype", [torch.bfloat16, torch.float32])
def test_gated_residual_rows(width, rows, branch_dtype):
    """Two streams of two batch items in one launch and each on its own, with and without the next norm."""
    g = torch.Generator(device=DEV).manual_seed(71)

    def randn(*shape, scale=1.0):
        return scale * torch.randn(*shape, generator=g, device=DEV)

    b = 2
    res = [randn(b, n, width) for n in rows]
    br = [randn(b, n, width).to(branch_dtype) for n in rows]
    w, w2 = ([1 + randn(width, scale=0.1) for _ in rows] for _ in range(2))
    gate, shift, scale = ([randn(b, 1, width, scale=0.1) for _ in rows] for _ in range(3))
    new = [r.double() + gt.double() * norm64(x, gw) for r, x, gt, gw in zip(res, br, gate, w)]
    nxt = [norm64(x, gw) * (1 + sc.double()) + sh.double() for x, gw, sc, sh in zip(new, w2, scale, shift)]
    for with_next in (False, True):
        got, one = ([r.clone() for r in res] for _ in range(2))
        outs, outs1 = ([torch.empty(r.shape, device=DEV) for r in res] for _ in range(2))
        tail = (w2, shift, scale, outs) if with_next else ()
        K.gated_residual_grouped_(got, br, w, gate, 1e-6, *tail)
        for i in range(2):
            if with_next:
                K.gated_residual_norm_modulate_(one[i], br[i], w[i], gate[i], 1e-6, w2[i], shift[i], scale[i], outs1[i])
                assert torch.equal(outs[i], outs1[i])
                torch.testing.assert_close(outs[i].double(), nxt[i], rtol=4e-6, atol=1e-5)
            else:
                K.gated_residual_rms_norm_(one[i], br[i], w[i], gate[i], 1e-6)
            assert torch.equal(got[i], one[i])
            torch.testing.assert_close(got[i].double(), new[i], rtol=2e-6, atol=4e-6)


@pytest.mark.parametrize("width", WIDTHS)
@pytest.mark.parametrize("rows", [1796, 1799])
def test_gated_residual_forms_agree(width, rows):
    """A launch past the split form's rows (with and without the coefficients shared by four rows)
    against its first rows alone."""
    g = torch.Generator(device=DEV).manual_seed(73)
    res, br = (torch.randn(1, rows, width, generator=g, device=DEV) for _ in range(2))
    br = br.to(torch.bfloat16)
    w, w2 = (1 + 0.1 * torch.randn(width, generator=g, device=DEV) for _ in range(2))
    gate, shift, scale = (0.1 * torch.randn(1, 1, width, generator=g, device=DEV) for _ in range(3))
    got, out = res.clone(), torch.empty(1, rows, width, device=DEV, dtype=torch.bfloat16)
    K.gated_residual_norm_modulate_(got, br, w, gate, 1e-6, w2, shift, scale, out)
    plain = K.gated_residual_rms_norm_(res.clone(), br, w, gate, 1e-6)
    assert torch.equal(plain, got)
    for n in (1, 333, 1790):
        part, part_out = res[:, :n].clone(), torch.empty(1, n, width, device=DEV, dtype=torch.bfloat16)
        K.gated_residual_norm_modulate_(part, br[:, :n].contiguous(), w, gate, 1e-6, w2, shift, scale, part_out)
        assert torch.equal(part, got[:, :n]) and torch.equal(part_out, out[:, :n])


@pytest.mark.parametrize("width", [*WIDTHS, 1408])
@pytest.mark.parametrize("rows,part", [((1412,), 1408), ((1411,), 1408), ((1200, 212), 1408)])
def test_gated_residual_forms_agree_around_the_shared_limit(width, rows, part):
    """With the next norm the wave form takes over earlier where four rows share its coefficients (1412
    rows, also of two streams) or a lane holds three chunks (1025 to 1536 columns): the same bits as the
    first 1408 rows in one launch."""
    g = torch.Generator(device=DEV).manual_seed(75)
    n = sum(rows)
    res, br = (torch.randn(1, n, width, generator=g, device=DEV) for _ in range(2))
    w, w2 = (1 + 0.1 * torch.randn(width, generator=g, device=DEV) for _ in range(2))
    gate, shift, scale = (0.1 * torch.randn(1, 1, width, generator=g, device=DEV) for _ in range(3))

    def run(*parts):
        r = [t.clone() for t in (res[:, a:b] for a, b in parts)]
        b = [br[:, a:b].contiguous() for a, b in parts]
        o = [torch.empty_like(t) for t in r]
        if len(parts) == 1:
            K.gated_residual_norm_modulate_(r[0], b[0], w, gate, 1e-6, w2, shift, scale, o[0])
        else:
            K.gated_residual_grouped_(r, b, [w] * 2, [gate] * 2, 1e-6, [w2] * 2, [shift] * 2, [scale] * 2, o)
        return torch.cat(r, 1), torch.cat(o, 1)

    whole = run((0, n)) if len(rows) == 1 else run((0, rows[0]), (rows[0], n))
    for got, want in zip(whole, run((0, part))):
        assert torch.equal(got[:, :part], want)


@pytest.mark.parametrize("width", [8, 264, *WIDTHS])
@pytest.mark.parametrize("rows", [1, 7, 130])
def test_residual_rms_norm_rows(width, rows):
    g = torch.Generator(device=DEV).manual_seed(72)
    res = torch.randn(rows, width, generator=g, device=DEV)
    w = 1 + 0.1 * torch.randn(width, generator=g, device=DEV)
    add = torch.randn(3, width, generator=g, device=DEV)
    for branch in (None, torch.randn(rows, width, generator=g, device=DEV).to(torch.bfloat16)):
        for extra in (None, add):
            r, out = res.clone(), torch.empty_like(res)
            K.residual_rms_norm(r, branch, w, 1e-6, out, add_rows=extra)
            new = res if branch is None else res + branch.float()
            assert torch.equal(r, new)
            want = norm64(new, w)
            if extra is not None:
                want = want + extra.double()[torch.arange(rows, device=DEV) % 3]
            torch.testing.assert_close(out.double(), want, rtol=2e-6, atol=4e-6)


@pytest.mark.parametrize("width", [128, 2560])
@pytest.mark.parametrize("batch,text,image", [(1, 3, 70), (2, 77, 240), (2, 1, 1000)])
def test_rows_enter_and_leave_a_residual_stream(width, batch, text, image):
    """``rms_norm_modulate_copy`` of text and image rows into one joined stream is the copies followed by
    ``rms_norm_modulate``; ``gated_residual_copy_`` is the residual followed by the copies (2 x 1001 rows:
    the wave form)."""
    g = torch.Generator(device=DEV).manual_seed(74)
    n = text + image
    rows = torch.randn(batch, n, width, generator=g, device=DEV)
    w = 1 + 0.1 * torch.randn(width, generator=g, device=DEV)
    shift, scale, gate = (0.1 * torch.randn(batch, 1, width, generator=g, device=DEV) for _ in range(3))
    stream = torch.full((batch * n, width), 5.0, device=DEV)
    h = torch.empty(batch * n, width, device=DEV, dtype=torch.bfloat16)
    K.rms_norm_modulate_copy(rows[:, :text].contiguous(), w, shift, scale, 1e-6, h, stream, n)
    K.rms_norm_modulate_copy(rows[:, text:].contiguous(), w, shift, scale, 1e-6, h, stream, n, text)
    assert torch.equal(stream.view(batch, n, width), rows)
    assert torch.equal(h.view(batch, n, width), K.rms_norm_modulate(rows, w, shift, scale, 1e-6, torch.bfloat16))
    want = K.gated_residual_rms_norm_(rows.clone(), h.view_as(rows), w, gate, 1e-6)
    first, rest = (torch.empty(batch, m, width, device=DEV) for m in (text, image))
    got, whole = stream.view(batch, n, width), torch.empty_like(rows)
    again = got.clone()
    K.gated_residual_copy_([got], [h.view_as(rows)], [w], [gate], 1e-6, [(first, rest)])
    assert torch.equal(got, want) and torch.equal(torch.cat([first, rest], 1), want)
    other = [again, rows[:, :text].contiguous()]
    K.gated_residual_copy_(other, [h.view_as(rows), h.view_as(rows)[:, :text].contiguous()], [w, w], [gate, gate], 1e-6,
                           (whole, first))
    assert torch.equal(again, want) and torch.equal(whole, want)
    assert torch.equal(other[1], want[:, :text]) and torch.equal(first, want[:, :text])
