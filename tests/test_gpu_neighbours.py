"""Parity of the path's neighbours (through the C ABI) against the CPU oracle:
the Linear layers of the time embedding, the row softmax, the DDIM schedule and
update.  Same criteria as test_gpu_parity.py; the DDIM update and everything
integer is bit-exact.
"""
import numpy as np
import pytest

from tolerances import assert_close_f16, assert_close_f32

pytestmark = pytest.mark.gpu


def _torch():
    import torch
    return torch


def _to_dev(a, cuda, half=False):
    t = _torch().from_numpy(np.ascontiguousarray(a)).to(cuda)
    return t.half() if half else t


# ----------------------------------------------------------------- Linear on embedding rows
def _linear_case(msd, orc, cuda, m, n, k, seed, half, act_in=0, act_out=0, bias=True):
    x = orc.normal((m, k), seed=seed)
    w = orc.normal((n, k), seed=seed + 1, sigma=1.0 / np.sqrt(k))
    b = orc.normal((n,), seed=seed + 2, sigma=0.1) if bias else None
    if half:
        x, w = orc.round_to_half(x), orc.round_to_half(w)
    xin = orc.silu(x) if act_in else x
    ref = orc.linear(xin, w, b)
    ref64 = orc.linear64(xin, w, b)
    if act_out:
        ref, ref64 = orc.silu(ref), orc.silu64(ref64.astype(np.float32))
    got = msd.linear_rows(_to_dev(x, cuda, half), _to_dev(w, cuda, half),
                          _to_dev(b, cuda) if bias else None, act_in, act_out).float().cpu().numpy()
    what = "linear m%d n%d k%d" % (m, n, k)
    if half:
        worst, exact = assert_close_f16(got, ref, what)
        return exact
    assert_close_f32(got, ref, what=what)
    if not act_out:
        assert_close_f32(got, ref64, 3e-6, what + " vs f64")
    return None


@pytest.mark.parametrize("name", ["lin_a", "lin_b", "lin_c"])
def test_linear_library_fixtures(msd, cuda, golden, name):
    x, w = golden[name + "_x"], golden[name + "_w"]
    b = _to_dev(golden[name + "_b"], cuda) if name + "_b" in golden.files else None
    xd, wd = _to_dev(x, cuda), _to_dev(w, cuda)
    assert_close_f32(msd.linear_rows(xd, wd, b).cpu().numpy(), golden[name + "_y"], what=name)
    assert_close_f32(msd.linear_rows(xd, wd, b, act_in=msd.ACT_SILU).cpu().numpy(),
                     golden[name + "_y_silu_in"], what=name + " silu in")
    assert_close_f32(msd.linear_rows(xd, wd, b, act_out=msd.ACT_SILU).cpu().numpy(),
                     golden[name + "_y_silu_out"], what=name + " silu out")


# time_embed_0 (320 -> 1280, SiLU behind it), time_embed_2 (1280 -> 1280), and the per-ResBlock
# SiLU(emb) -> Linear(1280 -> Cout) for Cout = 320 / 640 / 1280
@pytest.mark.parametrize("half", [False, True], ids=["f32", "f16"])
@pytest.mark.parametrize("n,k,act_in,act_out", [(1280, 320, 0, 1), (1280, 1280, 0, 0), (320, 1280, 1, 0),
                                                (640, 1280, 1, 0), (1280, 1280, 1, 0)])
def test_linear_time_embedding_shapes(msd, orc, cuda, n, k, act_in, act_out, half):
    exact = _linear_case(msd, orc, cuda, 2, n, k, 7000 + n + k, half, act_in, act_out)
    if half:
        assert exact > 0.99


@pytest.mark.parametrize("m,n,k", [(1, 64, 320), (3, 33, 96), (5, 7, 1280), (8, 130, 1280), (8, 16, 2048),
                                   (2, 5, 77), (4, 9, 1), (2, 3, 8), (7, 1, 40)])
def test_linear_edge_shapes(msd, orc, cuda, m, n, k):
    _linear_case(msd, orc, cuda, m, n, k, 7100 + m * 1000 + n + k, False)
    _linear_case(msd, orc, cuda, m, n, k, 7200 + m * 1000 + n + k, True, act_in=1, bias=False)


def test_linear_unaligned_views_and_rejections(msd, orc, cuda):
    torch = _torch()
    x = orc.normal((2, 328), seed=7301)
    w = orc.normal((20, 328), seed=7302, sigma=0.05)
    big = _to_dev(np.concatenate([[0.0], w.reshape(-1)]).astype(np.float32), cuda)
    wd = big[1:].view(20, 328)  # 4 bytes past a 16-byte boundary
    got = msd.linear_rows(_to_dev(x, cuda), wd).cpu().numpy()
    assert_close_f32(got, orc.linear(x, w), what="unaligned weight")
    lib = msd.load_library()
    xd = _to_dev(x, cuda)
    s = torch.cuda.current_stream().cuda_stream
    assert lib.msd_linear_rows(xd.data_ptr(), wd.data_ptr(), None, xd.data_ptr(), 2, 20, 328, 0, 0, 0, s) == 1
    nine = torch.zeros((9, 328), device=cuda)
    out = torch.zeros((9, 20), device=cuda)
    assert lib.msd_linear_rows(nine.data_ptr(), wd.data_ptr(), None, out.data_ptr(), 9, 20, 328, 0, 0, 0, s) == 1
    assert lib.msd_linear_rows(xd.data_ptr(), wd.data_ptr(), None, out.data_ptr(), 2, 20, 328, 2, 0, 0, s) == 1
    assert lib.msd_linear_rows(xd.data_ptr(), wd.data_ptr(), None, out.data_ptr(), 0, 20, 328, 0, 0, 0, s) == 0


# output channels of the 22 ResBlocks of one UNet step, in execution order (M/UNetModel.cpp:86-1018)
RESBLOCK_COUT = [320, 320, 640, 640, 1280, 1280, 1280, 1280, 1280, 1280, 1280, 1280, 1280, 1280, 1280, 1280,
                 640, 640, 640, 320, 320, 320]


@pytest.mark.parametrize("half", [False, True], ids=["f32", "f16"])
def test_grouped_linear_runs_the_22_resblock_projections_in_one_launch(msd, orc, cuda, half):
    """SiLU(emb) -> Linear(1280 -> Cout) of every ResBlock (M/nn/ResBlock.cpp:173-183) as one
    launch: each output against the oracle and bit for bit against its own msd_linear_rows call."""
    torch = _torch()
    emb = orc.normal((2, 1280), seed=7500, sigma=1.5)
    ws = [orc.normal((n, 1280), seed=7501 + i, sigma=1280 ** -0.5) for i, n in enumerate(RESBLOCK_COUT)]
    bs = [orc.normal((n,), seed=7601 + i, sigma=0.1) for i, n in enumerate(RESBLOCK_COUT)]
    if half:
        emb, ws = orc.round_to_half(emb), [orc.round_to_half(w) for w in ws]
    ed = _to_dev(emb, cuda, half)
    wd = [_to_dev(w, cuda, half) for w in ws]
    bd = [_to_dev(b, cuda) for b in bs]
    outs = msd.linear_rows_grouped(ed, wd, bd, act_in=msd.ACT_SILU)
    assert len(outs) == 22
    for i, (o, w, b) in enumerate(zip(outs, ws, bs)):
        single = msd.linear_rows(ed, wd[i], bd[i], act_in=msd.ACT_SILU)
        assert torch.equal(o, single), "problem %d differs from its own launch" % i
        ref = orc.linear(orc.silu(emb), w, b)
        if half:
            assert_close_f16(o.float().cpu().numpy(), ref, "grouped linear f16")
        else:
            assert_close_f32(o.cpu().numpy(), ref, what="grouped linear %d" % i)


@pytest.mark.parametrize("m", [3, 4, 5, 8])
@pytest.mark.parametrize("n,k", [(1, 640), (16, 648), (17, 704), (33, 1280), (15, 2568), (130, 4096), (7, 632)])
def test_linear_several_half_rows_on_the_matrix_cores(msd, orc, cuda, m, n, k):
    """Blocks of columns and rows with some left over; k of whole rounds of pieces, of cut ones, of more than one."""
    torch = _torch()
    for act_in, act_out, bias in ((0, 1, True), (1, 0, False), (1, 1, True)):
        _linear_case(msd, orc, cuda, m, n, k, 7950 + m + n + k, True, act_in, act_out, bias)
    x = orc.round_to_half(orc.normal((m, k), seed=7960 + k))
    w = orc.round_to_half(orc.normal((n, k), seed=7961 + k, sigma=k ** -0.5))
    xd, wd = _to_dev(x, cuda, True), _to_dev(w, cuda, True)
    single = msd.linear_rows(xd, wd, act_in=msd.ACT_SILU)
    other = _to_dev(orc.normal((9, k), seed=7962), cuda, True)
    for grouped in (msd.linear_rows_grouped(xd, [wd, other], act_in=msd.ACT_SILU)[0],
                    msd.linear_rows_grouped(xd, [other, wd], act_in=msd.ACT_SILU)[1]):
        assert torch.equal(grouped, single)


def test_linear_matrix_core_rows_with_infinities_nan_and_subnormals(msd, cuda):
    """An infinity or a NaN reaches the outputs it reaches in a sum of products, and no others; halves below the normal
    range count, in x, in the weights and in what SiLU leaves."""
    torch = _torch()
    g = torch.Generator(device=cuda).manual_seed(17)
    x = torch.randn((5, 1280), device=cuda, dtype=torch.float16, generator=g) + 0.25  # (no zeros: inf * 0)
    w = torch.randn((40, 1280), device=cuda, dtype=torch.float16, generator=g) * 0.03
    w[w == 0] = 0.01
    x[1, 700], x[2, 3], x[3, 1279] = float("inf"), float("nan"), -float("inf")
    w[5, 0], w[21, 650], w[39, 1279] = float("inf"), -float("inf"), float("nan")
    for act in (msd.ACT_NONE, msd.ACT_SILU):
        got = msd.linear_rows(x, w, act_in=act).double().cpu()
        xd, wd = x.double().cpu(), w.double().cpu()
        xd = xd / (1 + torch.exp(-xd)) if act else xd  # (-inf: NaN, as the product with 1 / (1 + inf))
        want = (xd[:, None, :] * wd[None]).sum(-1)
        assert torch.equal(torch.isnan(got), torch.isnan(want))
        assert torch.equal(torch.isinf(got), torch.isinf(want))
        assert torch.equal(got[torch.isinf(got)], want[torch.isinf(want)])
        fine = torch.isfinite(want)
        # half an ulp of the 16-bit result, and 1280 products' float32 sums
        assert float(((got - want)[fine].abs() / want[fine].abs().clamp(min=1.0)).max()) <= 2.0 ** -11 + 1e-5
    tiny = 2.0 ** -20  # x * w of halves below the normal range, against weights that bring the sum back
    xs = torch.full((4, 640), tiny, device=cuda, dtype=torch.float16)
    ws = torch.full((16, 640), 512.0, device=cuda, dtype=torch.float16)
    assert float((msd.linear_rows(xs, ws).double() - 640 * tiny * 512).abs().max()) <= 640 * tiny * 512 * 2.0 ** -11
    half_sum = 640 * 512 * (tiny / (1 + np.exp(-tiny)))
    assert float((msd.linear_rows(xs, ws, act_in=msd.ACT_SILU).double() - half_sum).abs().max()) <= half_sum * (2.0 ** -11 + 1e-5)
    assert float((msd.linear_rows(ws[:4], xs[:1]).double() - 640 * tiny * 512).abs().max()) <= 640 * tiny * 512 * 2.0 ** -11


@pytest.mark.parametrize("m", [3, 8])
@pytest.mark.parametrize("k", [640, 1288])
def test_linear_matrix_core_rows_keep_small_activated_values(msd, cuda, m, k):
    """What SiLU leaves of a row goes into the sum as a float32, however small it is: below the smallest half, and down to
    2^-38 at x = -30, against weights that bring the sum back into the range of halves."""
    torch = _torch()
    g = torch.Generator(device=cuda).manual_seed(31 + m + k)

    def check(x, w):
        x, w = x.to(torch.float16), w.to(torch.float16)
        got = msd.linear_rows(x, w, act_in=msd.ACT_SILU).double().cpu()
        xd = x.double().cpu()
        want = (xd / (1 + torch.exp(-xd))) @ w.double().cpu().t()
        assert float(want.abs().min()) > 2.0 ** -14  # (a normal half)
        # half an ulp of the result; SiLU's 2^x (1.2e-7 (1 + 1.45 |x|)) and float32 sums of k values of one sign
        assert float(((got - want) / want).abs().max()) <= 2.0 ** -11 + 2e-5
        grouped = msd.linear_rows_grouped(x, [w, w[:3]], act_in=msd.ACT_SILU)
        assert torch.equal(grouped[0].double().cpu(), got) and torch.equal(grouped[1].double().cpu(), got[:, :3])

    def uniform(rows, low, high):
        return torch.rand((rows, k), device=cuda, generator=g) * (high - low) + low

    for low, weight in ((-16.0, 100.0), (-20.0, 4e3), (-25.0, 6e4), (-27.0, 6e4), (-30.0, 6e4)):
        check(torch.full((m, k), low, device=cuda), torch.full((19, k), weight, device=cuda))
        check(uniform(m, low, low + 1), uniform(19, weight / 2, weight))
    for top in (-14, -18, -22):  # random magnitudes below 2^top, of both signs: SiLU halves them
        magnitude = uniform(m, 0.25, 1.0) * 2.0 ** top
        check(magnitude, uniform(19, 3e4, 6e4))
        check(-magnitude, uniform(19, 3e4, 6e4))
    # an infinite weight: a product with anything but zero is infinite, if its half would round to zero too
    for v in (-19.0, -21.0, -25.0, -40.0, -60.0, 2.0 ** -24, -2.0 ** -24):
        x = torch.full((m, k), v, device=cuda, dtype=torch.float16)
        w = torch.full((19, k), 0.5, device=cuda, dtype=torch.float16)
        w[0, 0], w[7, k - 1], w[18, k // 2] = float("inf"), -float("inf"), float("inf")
        got = msd.linear_rows(x, w, act_in=msd.ACT_SILU)
        sign = 1.0 if v > 0 else -1.0
        for col, inf in ((0, sign), (7, -sign), (18, sign)):
            assert bool((got[:, col] == inf * float("inf")).all()), v
        assert bool(torch.isfinite(got[:, [c for c in range(19) if c not in (0, 7, 18)]]).all())


@pytest.mark.parametrize("act_in", [0, 1])
@pytest.mark.parametrize("n,k", [(1, 8), (3, 120), (8, 128), (9, 136), (70, 512), (640, 504), (1283, 640), (1280, 1280),
                                 (33, 1288), (1281, 1544), (2563, 2568), (12289, 200), (12300, 1280)])
def test_linear_a_row_has_its_bits_alone_and_among_others(msd, cuda, n, k, act_in):
    """The sums of three to eight rows at once (four columns, and four or eight rows, per block of lanes; column quads, pieces
    and rounds left over) are those of a row by itself, a column or two per wavefront: the same products in the same order,
    with infinities, NaN and values of every size among them."""
    torch = _torch()
    g = torch.Generator(device=cuda).manual_seed(n + k)
    x = torch.randn((8, k), device=cuda, generator=g) * torch.logspace(-7, 4, 8, device=cuda)[:, None]
    x[3] = -torch.rand((k,), device=cuda, generator=g) * 100  # (SiLU leaves float32 values of 2^-143 and more)
    w = torch.randn((n, k), device=cuda, generator=g) * torch.logspace(-5, 3, n, device=cuda)[:, None]
    if n > 8:
        w[n - 1, k // 2], w[5, 0], x[6, k - 1] = float("inf"), -float("inf"), float("nan")
        x[1, 0], w[2, :8] = 0.0, 0.0
    x, w = x.to(torch.float16), w.to(torch.float16)
    bias = torch.randn((n,), device=cuda, generator=g)

    def bits(t):
        t = t.clone()
        t[t.isnan()] = float("nan")
        return t.view(torch.int16)

    for act_out in (0, 1):
        alone = torch.cat([msd.linear_rows(x[i:i + 1], w, bias, act_in=act_in, act_out=act_out) for i in range(8)])
        for m in (2, 3, 4, 5, 8):
            assert torch.equal(bits(msd.linear_rows(x[:m], w, bias, act_in=act_in, act_out=act_out)), bits(alone[:m]))
            grouped = msd.linear_rows_grouped(x[:m], [w[:1], w], [None, bias], act_in=act_in, act_out=act_out)[1]
            assert torch.equal(bits(grouped), bits(alone[:m]))


@pytest.mark.parametrize("m", [2, 3, 4, 5, 8])
@pytest.mark.parametrize("k", [4, 1280, 1284, 2564])
def test_large_grouped_linear_of_floats_is_each_layers_own(msd, cuda, m, k):
    """8192 columns and more of 4-byte weights share the rows in LDS: bit for bit what a column or two per wavefront
    give, with columns left over and k of one and of several chunks."""
    torch = _torch()
    g = torch.Generator(device=cuda).manual_seed(m * 10000 + k)
    x = torch.randn((m, k), device=cuda, generator=g)
    ws = [torch.randn((n, k), device=cuda, generator=g) * k ** -0.5 for n in (3, 8170, 1, 18)]
    bs = [torch.randn((w.shape[0],), device=cuda, generator=g) for w in ws]
    bs[2] = None
    for act_in, act_out in ((msd.ACT_SILU, msd.ACT_NONE), (msd.ACT_NONE, msd.ACT_SILU)):
        for out, w, b in zip(msd.linear_rows_grouped(x, ws, bs, act_in=act_in, act_out=act_out), ws, bs):
            assert torch.equal(out, msd.linear_rows(x, w, b, act_in=act_in, act_out=act_out))


def test_grouped_linear_edge_cases(msd, orc, cuda):
    torch = _torch()
    # more problems than one launch's table holds, empty problems, missing biases, no activation
    ns = [3, 0, 130, 1, 64] * 8
    x = orc.normal((3, 96), seed=7700)
    ws = [orc.normal((n, 96), seed=7701 + i, sigma=0.1) for i, n in enumerate(ns)]
    bs = [orc.normal((n,), seed=7801 + i) if i % 3 else None for i, n in enumerate(ns)]
    xd = _to_dev(x, cuda)
    outs = msd.linear_rows_grouped(xd, [_to_dev(w, cuda) for w in ws],
                                   [_to_dev(b, cuda) if b is not None else None for b in bs], act_out=msd.ACT_SILU)
    for o, w, b, n in zip(outs, ws, bs, ns):
        assert o.shape == (3, n)
        if n:
            assert_close_f32(o.cpu().numpy(), orc.silu(orc.linear(x, w, b)), what="grouped edge")
    # k that does not vectorise: falls back to one scalar launch per problem, same results
    x2 = orc.normal((2, 77), seed=7900)
    w2 = [orc.normal((5, 77), seed=7901), orc.normal((9, 77), seed=7902)]
    o2 = msd.linear_rows_grouped(_to_dev(x2, cuda), [_to_dev(w, cuda) for w in w2])
    for o, w in zip(o2, w2):
        assert_close_f32(o.cpu().numpy(), orc.linear(x2, w), what="grouped odd k")
    assert msd.linear_rows_grouped(xd, []) == []
    # rejections: more than 8 rows, an output that is the input
    lib = msd.load_library()
    import ctypes
    vp = ctypes.c_void_p
    arr = lambda *v: (vp * len(v))(*v)
    one = (ctypes.c_size_t * 1)(96)
    s = torch.cuda.current_stream().cuda_stream
    wdev = _to_dev(ws[2], cuda)
    assert lib.msd_linear_rows_grouped(xd.data_ptr(), arr(wdev.data_ptr()), None, arr(xd.data_ptr()), one, 1, 3, 96,
                                       0, 0, 0, s) == 1
    assert lib.msd_linear_rows_grouped(xd.data_ptr(), arr(wdev.data_ptr()), None, arr(outs[2].data_ptr()), one, 1, 9,
                                       96, 0, 0, 0, s) == 1


def test_time_embedding_mlp_chain(msd, orc, cuda):
    """timestep -> sinusoid -> Linear+SiLU -> Linear -> SiLU+Linear, as one UNet step runs it."""
    torch = _torch()
    t = np.array([981, 961], dtype=np.int64)
    w0 = orc.normal((1280, 320), seed=7401, sigma=320 ** -0.5)
    b0 = orc.normal((1280,), seed=7402, sigma=0.1)
    w2 = orc.normal((1280, 1280), seed=7403, sigma=1280 ** -0.5)
    b2 = orc.normal((1280,), seed=7404, sigma=0.1)
    we = orc.normal((640, 1280), seed=7405, sigma=1280 ** -0.5)
    be = orc.normal((640,), seed=7406, sigma=0.1)
    temb = np.stack([orc.timestep_embedding(int(v)) for v in t])
    h = orc.silu(orc.linear(temb, w0, b0))
    emb = orc.linear(h, w2, b2)
    ref = orc.linear(orc.silu(emb), we, be)
    d = lambda a: _to_dev(a, cuda)
    temb_d = msd.timestep_embedding(torch.from_numpy(t).to(cuda), 320)
    h_d = msd.linear_rows(temb_d, d(w0), d(b0), act_out=msd.ACT_SILU)
    emb_d = msd.linear_rows(h_d, d(w2), d(b2))
    out_d = msd.linear_rows(emb_d, d(we), d(be), act_in=msd.ACT_SILU)
    assert_close_f32(emb_d.cpu().numpy(), emb, what="time_embed")
    assert_close_f32(out_d.cpu().numpy(), ref, what="resblock emb projection")


# ----------------------------------------------------------------- softmax
def _softmax_case(msd, orc, cuda, rows, cols, seed, half, stable, sigma=2.0, inplace=False):
    x = orc.normal((rows, cols), seed=seed, sigma=sigma)
    if half:
        x = orc.round_to_half(x)
    ref = orc.softmax(x)
    xd = _to_dev(x, cuda, half)
    got = msd.softmax(xd, stable=stable, out=xd if inplace else None).float().cpu().numpy()
    what = "softmax %dx%d stable=%d" % (rows, cols, stable)
    if half:
        # probabilities are far below the 2e-3 absolute criterion: the stored value must be the
        # correct fp16 rounding of a value within 1e-5 RELATIVE of the oracle's
        worst, exact = assert_close_f16(got, ref, what, rel_floor=0.0)
        assert exact > 0.99, what
    else:
        assert_close_f32(got, ref, what=what)
        np.testing.assert_allclose(got, orc.softmax64(x), rtol=1e-5, atol=1e-9)
        np.testing.assert_allclose(got.astype(np.float64).sum(axis=-1), 1.0, atol=1e-5)


@pytest.mark.parametrize("stable", [0, 1])
@pytest.mark.parametrize("name", ["sm_a", "sm_b", "sm_c"])
def test_softmax_library_fixtures(msd, cuda, golden, name, stable):
    got = msd.softmax(_to_dev(golden[name + "_x"], cuda), stable=stable).cpu().numpy()
    assert_close_f32(got, golden[name + "_y"], what=name)
    np.testing.assert_allclose(got, golden[name + "_y"], rtol=1e-5, atol=1e-9)


# self-attention rows of the UNet (keys = 4096 / 1024 / 256 / 64 latent tokens) and the
# cross-attention rows (77 text tokens); rows cut down, the row length is what dispatches
@pytest.mark.parametrize("half", [False, True], ids=["f32", "f16"])
@pytest.mark.parametrize("stable", [0, 1])
@pytest.mark.parametrize("rows,cols", [(96, 4096), (130, 1024), (257, 256), (301, 64), (1000, 77)])
def test_softmax_attention_shapes(msd, orc, cuda, rows, cols, stable, half):
    _softmax_case(msd, orc, cuda, rows, cols, 8000 + cols, half, stable, inplace=True)


@pytest.mark.parametrize("rows,cols", [(1, 1), (3, 4), (5, 8), (9, 40), (7, 300), (4, 600), (6, 1000),
                                       (3, 2048), (5, 8192), (2, 10000), (33, 129), (2, 513),
                                       (200, 100), (128, 9), (64, 128), (191, 127), (70, 8),
                                       # rows of 3 ... 66 vectors: every team size of the register kernel,
                                       # row counts that leave part of the last wavefront without a row
                                       (67, 24), (35, 32), (50, 96), (45, 200), (21, 136), (19, 264)])
def test_softmax_edge_shapes(msd, orc, cuda, rows, cols):
    for half in (False, True):
        for stable in (0, 1):
            _softmax_case(msd, orc, cuda, rows, cols, 8100 + cols, half, stable, sigma=1.5)


@pytest.mark.parametrize("cols,half", [
    (129, True), (130, True), (252, True), (255, True), (257, True), (260, True), (324, True), (511, True), (513, True),
    (1023, True), (1026, True), (2044, True), (4095, True), (4097, True),
    (129, False), (130, False), (255, False), (257, False), (514, False), (1023, False), (2047, False), (2049, False)])
def test_softmax_rows_of_no_whole_vectors(msd, orc, cuda, cols, half):
    """Longer than the text scores, with every remainder of a vector around the steps of vectors per lane, up to
    the first row that goes to the kernel for any length."""
    for stable in (0, 1):
        _softmax_case(msd, orc, cuda, 11, cols, 7300 + cols + stable, half, stable, sigma=1.5, inplace=bool(stable))


@pytest.mark.parametrize("rows,cols,half", [
    (3071, 130, True), (3072, 130, True), (5119, 255, True), (5120, 255, True), (3075, 252, True), (8191, 260, True),
    (8195, 260, True), (8197, 511, True), (6143, 130, False), (8195, 254, False), (8195, 255, False), (8195, 510, False)])
def test_softmax_rows_of_no_whole_vectors_by_their_number(msd, orc, cuda, rows, cols, half):
    """On both sides of the numbers of rows from which 16-byte pieces replace single elements."""
    _softmax_case(msd, orc, cuda, rows, cols, 7500 + cols, half, rows % 2, sigma=1.5, inplace=True)


@pytest.mark.parametrize("cols,half", [
    (8200, True), (9216, True), (12288, True), (65536, True), (65544, True),       # 192, 192, 192, 1024 lanes; too long
    (4100, False), (8192, False), (8196, False), (12292, False), (16388, False), (32768, False), (32772, False)])
def test_softmax_rows_of_a_whole_workgroup(msd, orc, cuda, cols, half):
    """Rows longer than 1024 vectors: the shortest and the longest of each vectors-per-lane count
    and the first row that no workgroup holds."""
    for stable in (0, 1):
        _softmax_case(msd, orc, cuda, 5, cols, 8600 + cols + stable, half, stable, sigma=1.5, inplace=bool(stable))


@pytest.mark.parametrize("rows,cols,half", [
    (256, 2056, True), (257, 2056, True), (8191, 2056, True), (8192, 2560, True), (36864, 2568, True),   # wavefront or workgroup
    (45056, 2056, True), (40960, 4096, True), (16384, 4104, True), (8191, 8448, True), (8192, 9216, True),  # few rows open
    (256, 1028, False), (257, 4096, False), (3071, 1284, False), (3072, 1284, False), (45056, 1028, False),
    (8191, 5376, False), (8192, 5380, False), (8192, 8196, False)])
def test_softmax_long_rows_by_their_number(msd, orc, cuda, rows, cols, half):
    """On both sides of the numbers of rows at which a row gets a workgroup and the rows in flight are limited, with a
    vector more than each count of lanes holds; some rows of each launch, the first and the last among them."""
    torch = _torch()
    g = torch.Generator(device=cuda).manual_seed(rows + cols)
    x = torch.randn((rows, cols), device=cuda, dtype=torch.float16 if half else torch.float32, generator=g) * 1.5
    some = torch.tensor(sorted({0, 1, rows // 3, rows // 2 + 1, rows - 2, rows - 1}), device=cuda)
    ref = orc.softmax(x[some].float().cpu().numpy())
    for stable in (False, True):
        y = msd.softmax(x, stable=stable)
        got = y[some].float().cpu().numpy()
        if half:
            assert assert_close_f16(got, ref, "softmax, long rows", rel_floor=0.0)[1] > 0.99
        else:
            np.testing.assert_allclose(got, ref, rtol=1e-5, atol=1e-9)
        # every row was written: cols results of at most half an ulp of their size off (2^-11, and in 16-bit
        # storage the subnormal spacing 2^-25 each), and the sum's own rounding
        sums = y.sum(dim=-1, dtype=torch.float64)
        assert float((sums - 1.0).abs().max()) <= (2.0 ** -11 + cols * 2.0 ** -25 if half else 1e-5)
        del y, sums


@pytest.mark.parametrize("rb", [16, 32, 64])
def test_softmax_short_rows_flat_kernel(msd, orc, cuda, rb):
    """Rows of 77 / 100 moved as flat 16-byte vectors, rb rows per workgroup, plus a ragged tail."""
    lib = msd.load_library()
    assert lib.msd_set_tuning(msd.TUNE_SOFTMAX_ROWS, rb) == 0
    try:
        for rows, cols in [(rb * 5 + 3, 77), (rb, 100), (2 * rb + 1, 9), (rb * 3, 127)]:
            for half in (False, True):
                for stable in (0, 1):
                    _softmax_case(msd, orc, cuda, rows, cols, 8300 + cols + rb, half, stable, inplace=True)
    finally:
        assert lib.msd_set_tuning(msd.TUNE_SOFTMAX_ROWS, 0) == 0
    assert lib.msd_set_tuning(msd.TUNE_SOFTMAX_ROWS, 48) == 1


@pytest.mark.parametrize("rows,cols,half,knob", [
    (12288 + 7, 77, True, 0), (20000, 100, False, 0),    # 16 lanes per row, 32 / 16 rows per workgroup
    (40000 + 3, 77, False, 0), (40000, 100, True, 0),    # 8 lanes per row, 64 / 32 rows
    (66000 + 1, 77, True, 0), (66000, 100, True, 0),     # 4 lanes per row up to 80 columns, 8 beyond
    (66000, 77, False, 16), (66000, 33, True, 32), (40000, 127, True, 16), (40000, 9, False, 64)])
def test_softmax_flat_kernel_lanes_per_row(msd, orc, cuda, rows, cols, half, knob):
    """Row counts on both sides of the limits where the flat kernel changes its lanes per row."""
    lib = msd.load_library()
    assert lib.msd_set_tuning(msd.TUNE_SOFTMAX_ROWS, knob) == 0
    try:
        for stable in (0, 1):
            _softmax_case(msd, orc, cuda, rows, cols, 8500 + cols + stable, half, stable, inplace=bool(stable))
    finally:
        assert lib.msd_set_tuning(msd.TUNE_SOFTMAX_ROWS, 0) == 0


def test_softmax_cross_attention_full_rows(msd, orc, cuda):
    """All 2 x 8 x 4096 query rows against 77 text tokens (the size that takes the flat kernel)."""
    _softmax_case(msd, orc, cuda, 2 * 8 * 4096, 77, 8400, True, 0, inplace=True)
    _softmax_case(msd, orc, cuda, 2 * 8 * 4096 + 5, 77, 8401, False, 1)


def test_softmax_overflow_follows_the_reference_unless_stable(msd, orc, cuda):
    x = np.zeros((2, 64), dtype=np.float32)
    x[0, 1], x[0, 2] = 89.0, 1.0
    x[1, :] = np.linspace(-3, 3, 64)
    with np.errstate(all="ignore"):
        ref = orc.softmax(x)
    got = msd.softmax(_to_dev(x, cuda), stable=False).cpu().numpy()
    assert np.isnan(ref[0, 1]) and np.isnan(got[0, 1])
    assert got[0, 0] == 0.0 and got[0, 2] == 0.0
    assert_close_f32(got[1], ref[1], what="finite row next to an overflowing one")
    safe = msd.softmax(_to_dev(x, cuda), stable=True).cpu().numpy()
    np.testing.assert_allclose(safe, orc.softmax64(x), rtol=1e-5, atol=1e-30)


def test_softmax_full_size_rows_sum_to_one(msd, cuda):
    """One attention map of the first UNet level at full size: 8 heads x 4096 x 4096, fp16, in place."""
    torch = _torch()
    g = torch.Generator(device=cuda)
    g.manual_seed(8200)
    x = torch.randn((8 * 4096, 4096), device=cuda, dtype=torch.float16, generator=g) * 3.0
    keep = x[:64].float().cpu().numpy()
    msd.softmax(x, stable=False, out=x)
    sums = x.float().sum(dim=-1)
    assert float((sums - 1.0).abs().max()) < 2e-2  # 4096 values rounded to fp16 each
    assert float(x.min()) >= 0.0 and float(x.max()) <= 1.0
    e = np.exp(keep.astype(np.float64))
    assert_close_f16(x[:64].float().cpu().numpy(), e / e.sum(axis=-1, keepdims=True), "softmax 65536x4096, 64 rows",
                     rel_floor=0.0)


# ----------------------------------------------------------------- DDIM
def test_ddim_schedule_is_bit_exact(msd, orc):
    assert np.array_equal(np.asarray(msd.alphas_cumprod(), dtype=np.float32), orc.alphas_cumprod())
    for steps in (50, 25, 30, 7, 1, 500):
        got, ref = msd.ddim_schedule(steps), orc.ddim_schedule(steps)
        for g, r in zip(got, ref):
            assert np.array_equal(np.asarray(g, dtype=r.dtype), r)
    lib = msd.load_library()
    assert lib.msd_ddim_schedule(0, None, None, None, None, 0) == -1
    assert lib.msd_ddim_schedule(501, None, None, None, None, 0) == -2


@pytest.mark.parametrize("n", [4 * 64 * 64, 2 * 4 * 64 * 64, 1001, 3, 1])
def test_ddim_update_fp32_is_bit_exact(msd, orc, cuda, n):
    x = orc.normal((n,), seed=9000 + n)
    e = orc.normal((n,), seed=9100 + n)
    ts, a, ap, s1m = orc.ddim_schedule(50)
    for index in (49, 30, 0):
        ref = orc.ddim_update(x, e, a[index], ap[index], s1m[index])
        xd = _to_dev(x, cuda)
        got = msd.ddim_update(xd, _to_dev(e, cuda), float(a[index]), float(ap[index]), float(s1m[index]))
        assert np.array_equal(got.cpu().numpy(), ref)
        msd.ddim_update(xd, _to_dev(e, cuda), float(a[index]), float(ap[index]), float(s1m[index]), out=xd)
        assert np.array_equal(xd.cpu().numpy(), ref)


def test_ddim_update_fixture_unaligned_and_fp16(msd, orc, cuda, golden):
    x, e = golden["ddim_x"], golden["ddim_e"]
    a_t, a_prev = np.float32(golden["ddim_a_t"]), np.float32(golden["ddim_a_prev"])
    s1m = np.sqrt(np.float32(1.0) - a_t)
    got = msd.ddim_update(_to_dev(x, cuda), _to_dev(e, cuda), float(a_t), float(a_prev), float(s1m))
    assert_close_f32(got.cpu().numpy(), golden["ddim_x_prev_f64"], 2e-6, "ddim vs LDM f64")
    xo = _to_dev(np.concatenate([[0.0], x]).astype(np.float32), cuda)[1:]
    eo = _to_dev(np.concatenate([[0.0], e]).astype(np.float32), cuda)[1:]
    got = msd.ddim_update(xo, eo, float(a_t), float(a_prev), float(s1m))
    assert np.array_equal(got.cpu().numpy(), orc.ddim_update(x, e, a_t, a_prev, s1m))
    xh, eh = orc.round_to_half(x), orc.round_to_half(e)
    goth = msd.ddim_update(_to_dev(xh, cuda, True), _to_dev(eh, cuda, True), float(a_t), float(a_prev), float(s1m))
    ref16 = orc.round_to_half(orc.ddim_update(xh, eh, a_t, a_prev, s1m))
    assert np.array_equal(goth.float().cpu().numpy(), ref16)  # same float32 value, rounded once


def test_ddim_sampling_loop_is_bit_exact(msd, orc, cuda):
    """25 steps, walked from the back as the sampler does, with a stand-in noise model."""
    ts, a, ap, s1m = orc.ddim_schedule(25)
    x = orc.normal((4 * 64 * 64,), seed=9201)
    noise = orc.normal((4 * 64 * 64,), seed=9202)
    xd, nd = _to_dev(x, cuda), _to_dev(noise, cuda)
    for index in range(len(ts) - 1, -1, -1):
        scale = np.float32(0.25 + 0.001 * ts[index])
        e = (np.float32(0.5) * x + scale * noise).astype(np.float32)
        ed = xd * 0.5 + nd * float(scale)  # torch float32 elementwise: same roundings as numpy
        x = orc.ddim_update(x, e, a[index], ap[index], s1m[index])
        msd.ddim_update(xd, ed, float(a[index]), float(ap[index]), float(s1m[index]), out=xd)
    assert np.array_equal(xd.cpu().numpy(), x)


@pytest.mark.parametrize("rows,cols,half", [(70, 256, True), (3075, 256, True), (9, 1024, True), (70, 256, False), (9, 1024, False),
                                            (5, 2048, False)])
def test_softmax_rows_that_start_at_any_element(msd, orc, cuda, rows, cols, half):
    """Whole vectors in length, one element past an aligned address; nothing is written around the output."""
    torch = _torch()
    n = rows * cols
    x = orc.normal((rows, cols), seed=8700 + cols, sigma=1.5)
    x = orc.round_to_half(x) if half else x
    buf = torch.full((n + 2,), 7.0, dtype=torch.float16 if half else torch.float32, device=cuda)
    buf[1:n + 1] = _to_dev(x, cuda, half).reshape(-1)
    at = buf.data_ptr() + buf.element_size()
    assert msd.load_library().msd_softmax(at, at, rows, cols, 1, msd.DTYPE_F16 if half else msd.DTYPE_F32, None) == 0
    torch.cuda.synchronize()
    got = buf.float().cpu().numpy()
    assert got[0] == 7.0 and got[n + 1] == 7.0
    got = got[1:n + 1].reshape(rows, cols)
    if half:
        assert assert_close_f16(got, orc.softmax(x), "softmax, unaligned rows", rel_floor=0.0)[1] > 0.99
    else:
        np.testing.assert_allclose(got, orc.softmax64(x), rtol=1e-5, atol=1e-9)


@pytest.mark.parametrize("cols,rows,half", [(9216, 8, True), (8196, 8, False),              # a workgroup's registers
                                            (252, 3080, True), (514, 8, True), (1023, 8, False),   # pieces, cut ones too
                                            (147, 8, True), (255, 8, False)])                    # single elements
def test_softmax_rows_with_infinities_and_nan(msd, cuda, cols, rows, half):
    """Masked positions are 0; a row of -inf, or with +inf or NaN, is NaN throughout where the maximum is taken
    first (0 / 0 and inf - inf), and never touches its neighbours."""
    torch = _torch()
    x = torch.empty((rows, cols), device=cuda).normal_(0.0, 1.5)
    x = (x.half() if half else x)
    x[0, cols // 2:] = -float("inf")
    x[1] = -float("inf")
    x[2, cols - 1] = float("inf")
    x[3, 0] = float("nan")
    x[4, 1:] = torch.finfo(x.dtype).min
    x[5] = -65504.0
    ref = torch.softmax(x.double().cpu(), -1)
    for inplace in (False, True):
        y = x.clone()
        got = msd.softmax(y, stable=True, out=y if inplace else None).double().cpu()
        for i in range(rows):
            assert torch.equal(torch.isnan(got[i]), torch.isnan(ref[i])), (i, inplace)
        ok = ~torch.isnan(ref)
        assert (got[0, cols // 2:] == 0).all()
        # half an ulp of the stored value (2^-11 of it in fp16, 2^-25 below the normal range) and 1e-5 of it
        torch.testing.assert_close(got[ok], ref[ok], rtol=1e-5 + (2.0 ** -11 if half else 0.0), atol=2.0 ** -25 if half else 1e-9)
    with_mask = msd.softmax(x[:1].clone(), stable=False).double().cpu()
    torch.testing.assert_close(with_mask, ref[:1], rtol=1e-5 + (2.0 ** -11 if half else 0.0), atol=2.0 ** -25 if half else 1e-9)
