"""The two additions the reference runs in front of its norms (chunkwise_add before the
ResBlock out-norm, elemwise_add before LayerNorm 2 / 3) and their fusion into the norm
kernels.  Fused launches must equal the two-launch sequence bit for bit, and both must match
the CPU oracle's restatement of the reference kernels."""
import ctypes

import numpy as np
import pytest

from tolerances import assert_close_f16, assert_close_f32, assert_one_ulp16_apart

pytestmark = pytest.mark.gpu


def _dev(a, cuda, half=False):
    import torch
    t = torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
    return t.half() if half else t


def _affine(orc, n, seed):
    return (orc.normal((n,), seed=seed, mean=1.0, sigma=0.1), orc.normal((n,), seed=seed + 1, sigma=0.1))


@pytest.mark.parametrize("half", [False, True], ids=["f32", "f16"])
@pytest.mark.parametrize("n,chunk", [(2 * 320 * 1024, 1024), (3 * 7 * 9, 9), (1031, 0), (2 * 4096 * 320, 0), (40, 8)])
def test_add_kernels(msd, orc, cuda, n, chunk, half):
    a = orc.normal((n,), seed=n, sigma=2.0)
    if chunk:
        b = orc.normal((n // chunk,), seed=n + 1)
    else:
        b = orc.normal((n,), seed=n + 1)
    ain, bin_ = (orc.round_to_half(a), orc.round_to_half(b)) if half else (a, b)
    ref = orc.chunkwise_add(ain, bin_, chunk) if chunk else orc.elemwise_add(ain, bin_)
    ad, bd = _dev(ain, cuda, half), _dev(bin_, cuda, half)
    got = msd.chunkwise_add(ad, bd, chunk, out=ad) if chunk else msd.elemwise_add(ad, bd, out=ad)  # in place
    got = got.float().cpu().numpy()
    if half:
        assert np.array_equal(got, orc.round_to_half(ref))  # one rounding of an exact sum
    else:
        assert np.array_equal(got, ref)


@pytest.mark.parametrize("half,shape,vectors", [
    (True, (32, 640, 600), 6), (True, (24, 256, 1536), 6), (False, (32, 640, 300), 6), (False, (24, 128, 1536), 6),
    (False, (32, 64, 500), 1), (False, (48, 256, 304), 3), (False, (32, 64, 2560), 5), (False, (28, 128, 836), 4)])
def test_chunk_add_groupnorm_of_several_workgroups_per_cu(msd, orc, cuda, half, shape, vectors):
    """Slices that fill their vectors in every lane and slices that do not, of launches that ask for gamma and beta behind the data."""
    import torch
    batch, channels, hw = shape
    assert msd.groupnorm_plan(batch, channels, hw, 32, msd.DTYPE_F16 if half else msd.DTYPE_F32)[1:3] == (256, vectors)
    x = orc.normal(shape, seed=hw, sigma=1.5, mean=0.3)
    emb = orc.normal((batch, channels), seed=hw + 1, sigma=0.7)
    g, b = _affine(orc, channels, 9)
    x, emb = (orc.round_to_half(x), orc.round_to_half(emb)) if half else (x, emb)
    xd, ed, gd, bd = _dev(x, cuda, half), _dev(emb, cuda, half), _dev(g, cuda), _dev(b, cuda)
    for silu in (True, False):
        tmp = msd.chunkwise_add(xd, ed, hw)
        two = msd.groupnorm(tmp, gd, bd, 32, 1e-5, silu)
        assert torch.equal(msd.chunk_add_groupnorm(xd, ed, gd, bd, 32, 1e-5, silu), two)
        ref = orc.groupnorm64(tmp.float().cpu().numpy(), g, b, 32, 1e-5, silu).astype(np.float32).reshape(shape)
        (assert_close_f16 if half else assert_close_f32)(two.float().cpu().numpy(), ref, what="several workgroups per CU")


@pytest.mark.parametrize("half", [False, True], ids=["f32", "f16"])
@pytest.mark.parametrize("shape,groups", [((2, 320, 64, 64), 32), ((2, 640, 32, 32), 32), ((2, 1280, 8, 8), 32),
                                          ((1, 96, 24, 24), 32), ((3, 64, 5, 7), 8), ((1, 8, 128, 128), 1)])
def test_chunk_add_groupnorm_equals_two_launches(msd, orc, cuda, shape, groups, half):
    import torch
    batch, channels = shape[0], shape[1]
    hw = int(np.prod(shape[2:]))
    x = orc.normal(shape, seed=sum(shape), sigma=1.5)
    emb = orc.normal((batch, channels), seed=sum(shape) + 1, sigma=0.7)
    g, b = _affine(orc, channels, 7)
    xin, ein = (orc.round_to_half(x), orc.round_to_half(emb)) if half else (x, emb)
    xd, ed, gd, bd = _dev(xin, cuda, half), _dev(ein, cuda, half), _dev(g, cuda), _dev(b, cuda)
    fused = msd.chunk_add_groupnorm(xd, ed, gd, bd, groups, 1e-5, True)
    tmp = msd.chunkwise_add(xd, ed, hw)
    two = msd.groupnorm(tmp, gd, bd, groups, 1e-5, True)
    assert torch.equal(fused, two)
    # in place, as the reference runs its out-norm (M/nn/ResBlock.cpp:222): the launch never lets
    # several workgroups share a unit then, so it is compared with the same launch out of place
    lib = msd.load_library()
    assert lib.msd_set_tuning(msd.TUNE_GN_WRITERS, 1) == 0
    try:
        apart = msd.chunk_add_groupnorm(xd.clone(), ed, gd, bd, groups, 1e-5, True)
    finally:
        assert lib.msd_set_tuning(msd.TUNE_GN_WRITERS, 0) == 0
    xc = xd.clone()
    assert torch.equal(msd.chunk_add_groupnorm(xc, ed, gd, bd, groups, 1e-5, True, out=xc), apart)
    # oracle: chunkwise_add, (storage rounding), group norm, silu
    s = orc.chunkwise_add(xin, ein, hw)
    if half:
        s = orc.round_to_half(s)
    ref = orc.groupnorm64(s, g, b, groups, 1e-5, True)
    got = fused.float().cpu().numpy()
    if half:
        assert_close_f16(got, ref.astype(np.float32), "chunk add gn f16")
    else:
        assert_close_f32(got, ref, what="chunk add gn f32")
    assert msd.status() == 0


@pytest.mark.parametrize("batch,channels,hw,groups,half", [
    (2, 1280, 63, 32, True), (2, 2560, 63, 32, True), (1, 2560, 81, 32, False),   # the deepest level: odd sizes, shared units
    (2, 640, 252, 32, True), (20, 1280, 252, 32, True),                           # multiples of four: shared, whole units
    (2, 320, 4092, 32, True), (1, 320, 16380, 32, True), (1, 320, 16390, 32, False),  # slices, the last one shorter
    (1, 80, 9, 2, True), (3, 32, 5, 4, False), (2, 64, 8 + 1, 8, True),           # barely a vector per channel
    (1, 16, 7, 2, True), (1, 24, 63, 8, True),                                    # below it; units of no whole vectors
    (2, 8, 40961, 1, True)])                                                      # slices that start inside a channel
def test_groupnorm_channels_of_no_whole_vectors(msd, orc, cuda, batch, channels, hw, groups, half):
    """Vectors that hold the end of one channel and the start of the next, with and without the
    addend, SiLU and a large mean, apart and in place."""
    import torch
    x = orc.normal((batch, channels, hw), seed=channels + hw, sigma=1.5)
    emb = orc.normal((batch, channels), seed=channels + hw + 1, sigma=0.7)
    g, b = _affine(orc, channels, 11)
    xin, ein = (orc.round_to_half(x), orc.round_to_half(emb)) if half else (x, emb)
    gd, bd, ed = _dev(g, cuda), _dev(b, cuda), _dev(ein, cuda, half)
    close = assert_close_f16 if half else assert_close_f32
    for mean, silu in ((0.0, True), (9.0, False)):  # 9: the mean is not folded into the offset
        shifted = orc.round_to_half(xin + mean) if half else (xin + mean).astype(np.float32)
        ref = orc.groupnorm64(shifted, g, b, groups, 1e-5, silu).astype(np.float32)
        for inplace in (False, True):
            xd = _dev(shifted, cuda, half)
            got = msd.groupnorm(xd, gd, bd, groups, 1e-5, silu, out=xd if inplace else None)
            close(got.float().cpu().numpy(), ref, what="gn ragged")
            xd = _dev(shifted, cuda, half)
            apart = torch.empty_like(xd)
            tmp = msd.chunkwise_add(xd, ed, hw)
            two = msd.groupnorm(tmp, gd, bd, groups, 1e-5, silu, out=tmp if inplace else apart)
            fused = msd.chunk_add_groupnorm(xd, ed, gd, bd, groups, 1e-5, silu, out=xd if inplace else None)
            assert torch.equal(fused, two)
    assert msd.status() == 0


@pytest.mark.parametrize("half", [False, True], ids=["f32", "f16"])
@pytest.mark.parametrize("rows,dim", [(8192, 320), (2048, 640), (512, 1280), (77, 1024), (5, 100), (9, 64)])
def test_add_layernorm_equals_two_launches(msd, orc, cuda, rows, dim, half):
    import torch
    a = orc.normal((rows, dim), seed=rows + dim, sigma=1.2)
    r = orc.normal((rows, dim), seed=rows + dim + 1, sigma=0.8, mean=0.5)
    g, b = _affine(orc, dim, 9)
    ain, rin = (orc.round_to_half(a), orc.round_to_half(r)) if half else (a, r)
    ad, rd, gd, bd = _dev(ain, cuda, half), _dev(rin, cuda, half), _dev(g, cuda), _dev(b, cuda)
    s_fused, y_fused = msd.add_layernorm(ad, rd, gd, bd)
    s_two = msd.elemwise_add(ad, rd)
    y_two = msd.layernorm(s_two, gd, bd)
    assert torch.equal(s_fused, s_two) and torch.equal(y_fused, y_two)
    # sum written over the first operand, as M/nn/BasicTransformerBlock.cpp:126-134 does
    ac = ad.clone()
    s_in, y_in = msd.add_layernorm(ac, rd, gd, bd, sum_out=ac)
    assert s_in.data_ptr() == ac.data_ptr() and torch.equal(s_in, s_two) and torch.equal(y_in, y_two)
    s_ref = orc.elemwise_add(ain, rin)
    if half:
        s_ref = orc.round_to_half(s_ref)
    ref = orc.layernorm64(s_ref, g, b, 1e-5)
    got = y_fused.float().cpu().numpy()
    if half:
        assert np.array_equal(s_fused.float().cpu().numpy(), s_ref)
        assert_close_f16(got, ref.astype(np.float32), "add ln f16")
    else:
        assert np.array_equal(s_fused.cpu().numpy(), s_ref)
        assert_close_f32(got, ref, what="add ln f32")


@pytest.mark.parametrize("half", [False, True], ids=["f32", "f16"])
@pytest.mark.parametrize("shape,groups,split", [((2, 320, 64, 64), 32, 0), ((2, 640, 32, 32), 32, 0),
                                                ((2, 1280, 16, 16), 32, 0), ((2, 1280, 8, 8), 32, 0),
                                                ((1, 320, 64, 64), 32, 8), ((2, 640, 32, 32), 32, 2),
                                                ((1, 96, 24, 24), 32, 0), ((3, 64, 5, 7), 8, 0),
                                                ((1, 33, 4, 4), 33, 0), ((1, 8, 128, 128), 1, 0),
                                                ((8, 320, 32, 32), 32, 0), ((4, 640, 32, 32), 32, 0)])
@pytest.mark.parametrize("writers", [0, 1, 4, 16], ids=["writers-auto", "one-writer", "4-writers", "16-writers"])
def test_groupnorm_tokens_equals_norm_then_permute(msd, orc, cuda, shape, groups, split, half, writers):
    """SpatialTransformer's GroupNorm(eps 1e-6, no SiLU) + permute (0, 2, 1) in one launch
    (M/nn/SpatialTransformer.cpp:127-139): slices of positions with an exchange, or (writers != 1,
    where the shape allows it) several workgroups that each reduce the whole unit and store the
    tokens of one range of positions."""
    import torch
    lib = msd.load_library()
    batch, channels = shape[0], shape[1]
    hw = int(np.prod(shape[2:]))
    x = orc.normal(shape, seed=sum(shape) + 3, sigma=1.5, mean=0.4)
    g, b = _affine(orc, channels, 11)
    xin = orc.round_to_half(x) if half else x
    xd, gd, bd = _dev(xin, cuda, half), _dev(g, cuda), _dev(b, cuda)
    try:
        lib.msd_set_tuning(msd.TUNE_GN_SPLIT, split)
        assert lib.msd_set_tuning(msd.TUNE_GN_WRITERS, writers) == 0
        fused = msd.groupnorm_tokens(xd, gd, bd, groups, 1e-6)
    finally:
        lib.msd_set_tuning(msd.TUNE_GN_SPLIT, 0)
        lib.msd_set_tuning(msd.TUNE_GN_WRITERS, 0)
    two = msd.groupnorm(xd, gd, bd, groups, 1e-6, False).view(batch, channels, hw).permute(0, 2, 1).contiguous()
    assert fused.shape == (batch, hw, channels)
    # the slices cut positions instead of channel ranges, so the statistics are summed in another
    # order: equal to the two-launch result up to that (a few float ulps), not bit for bit
    d = (fused.float() - two.float()).abs()
    if half:
        assert (d == 0).float().mean().item() > 0.999
        assert_one_ulp16_apart(fused.float().cpu().numpy(), two.float().cpu().numpy(), "gn tokens vs two launches")
    else:
        assert (d / two.abs().clamp(min=1.0)).max().item() < 2e-6
    ref = np.concatenate([orc.permute_0_2_1(orc.groupnorm64(xin, g, b, groups, 1e-6, False)
                                            .astype(np.float32).reshape(batch, channels, hw)[i:i + 1])
                          for i in range(batch)])
    got = fused.float().cpu().numpy()
    if half:
        assert_close_f16(got, ref, "gn tokens f16")
    else:
        assert_close_f32(got, ref, what="gn tokens f32")
    assert msd.status() == 0


@pytest.mark.parametrize("mean", [0.4, 60.0], ids=["", "far-mean"])  # 60: the statistics take their second pass
@pytest.mark.parametrize("shape,groups,half", [
    ((2, 640, 36, 28), 32, True), ((2, 640, 24, 24), 32, True), ((1, 1280, 24, 24), 32, True),  # parts of unequal length
    ((2, 640, 32, 32), 32, False), ((3, 320, 10, 8), 32, False), ((1, 1280, 16, 8), 32, False),
    ((2, 1280, 18, 14), 32, True), ((5, 1280, 18, 22), 32, True), ((9, 640, 6, 10), 32, True),  # vectors across channels
    ((1, 1280, 2, 2), 32, True), ((3, 136, 6, 6), 17, True), ((3, 136, 6, 6), 17, False),       # rows of half a vector; 17 groups
    ((16, 64, 16, 16), 32, True), ((7, 96, 4, 4), 96, False), ((33, 64, 8, 8), 32, True),       # one word per position; odd batches
    ((5, 1280, 28, 28), 32, True), ((1, 1280, 40, 40), 32, True)])                              # a part more for the LDS; long units
def test_groupnorm_tokens_of_whole_units(msd, orc, cuda, shape, groups, half, mean):
    """One launch in which every workgroup reduces whole units: against the oracle in 64 bits, eagerly and recorded."""
    import torch
    batch, channels, hw = shape[0], shape[1], shape[2] * shape[3]
    x = orc.normal(shape, seed=sum(shape) + 9, sigma=1.5, mean=mean)
    g, b = _affine(orc, channels, 27)
    xin = orc.round_to_half(x) if half else x
    ref = orc.groupnorm64(xin, g, b, groups, 1e-6, False).astype(np.float32).reshape(batch, channels, hw).transpose(0, 2, 1)
    xd, gd, bd = _dev(xin, cuda, half), _dev(g, cuda), _dev(b, cuda)
    assert not _takes_two_launches(msd, xd, gd, bd, groups)
    eager = msd.groupnorm_tokens(xd, gd, bd, groups, 1e-6)
    (assert_close_f16 if half else assert_close_f32)(eager.float().cpu().numpy(), ref, what="gn tokens, whole units")
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.graph(graph, stream=stream):
        recorded = msd.groupnorm_tokens(xd, gd, bd, groups, 1e-6)
    for _ in range(3):
        recorded.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(recorded, eager)


@pytest.mark.parametrize("shape", [(2, 320, 71, 70),                        # cut into slices outside a capture; whole in it
                                   (2, 640, 63, 63), (1, 640, 127, 65)])    # longer than one workgroup holds
def test_groupnorm_of_no_whole_vectors_is_recorded_without_scratch(msd, orc, cuda, shape):
    """A stream that has no scratch and is being captured, where none can be made."""
    import torch
    x = orc.normal(shape, seed=sum(shape), sigma=1.5)
    g, b = _affine(orc, shape[1], 31)
    xd, gd, bd = _dev(x, cuda), _dev(g, cuda), _dev(b, cuda)
    ref = orc.groupnorm64(x.reshape(shape[0], shape[1], -1), g, b, 32, 1e-5, True).astype(np.float32).reshape(shape)
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    assert msd.load_library().msd_release(stream.cuda_stream) == 0  # (an earlier stream may have had this handle)
    with torch.cuda.graph(graph, stream=stream):
        recorded = msd.groupnorm(xd, gd, bd, 32, 1e-5, True)
    for _ in range(3):
        recorded.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert_close_f32(recorded.cpu().numpy(), ref, what="gn ragged, recorded without scratch")


@pytest.mark.parametrize("shape,half,plan", [
    ((1, 128, 512, 512), False, (32, 512, 16)), ((1, 128, 512, 512), True, (16, 512, 16)),  # the whole 512 lanes
    ((1, 512, 192, 192), False, (32, 512, 10)),                                            # 4608 vectors a slice
    ((1, 128, 320, 392), False, (16, 512, 16)),                                            # 7840: masked lanes
    ((9, 64, 192, 384), True, (4, 512, 10)),                                               # halves, then quarters
    ((1, 128, 384, 384), True, (8, 960, 10))])                                             # one per CU, not longer than 12288: stays
def test_groupnorm_long_slices_are_cut_for_512_lanes(msd, orc, cuda, shape, half, plan):
    x = orc.normal(shape, seed=sum(shape), sigma=1.5, mean=0.3)
    g, b = _affine(orc, shape[1], 41)
    got_plan = msd.groupnorm_plan(shape[0], shape[1], shape[2] * shape[3], 32, msd.DTYPE_F16 if half else msd.DTYPE_F32)
    assert got_plan[:3] == plan and got_plan[3] == 1
    xin = orc.round_to_half(x) if half else x
    ref = orc.groupnorm64(xin, g, b, 32, 1e-6, True).astype(np.float32)
    xd, gd, bd = _dev(xin, cuda, half), _dev(g, cuda), _dev(b, cuda)
    apart = msd.groupnorm(xd, gd, bd, 32, 1e-6, True).float().cpu().numpy()
    inplace = msd.groupnorm(xd, gd, bd, 32, 1e-6, True, out=xd).float().cpu().numpy()
    (assert_close_f16 if half else assert_close_f32)(apart, ref, what="gn, long slices")
    assert np.array_equal(apart, inplace)


def _takes_two_launches(msd, xd, gd, bd, groups):
    """Only two launches leave anything in the workspace."""
    import torch
    batch, channels = xd.shape[:2]
    workspace = torch.zeros(batch * groups * msd.TOKENS_WORKSPACE_BYTES, dtype=torch.uint8, device=xd.device)
    out = torch.empty_like(xd)
    assert msd.load_library().msd_groupnorm_tokens_workspace(
        xd.data_ptr(), out.data_ptr(), gd.data_ptr(), bd.data_ptr(), batch, channels, xd.numel() // (batch * channels), groups,
        1e-6, msd.DTYPE_F16 if xd.dtype == torch.float16 else msd.DTYPE_F32, workspace.data_ptr(), workspace.numel(),
        torch.cuda.current_stream().cuda_stream) == 0
    return bool(workspace.any())


@pytest.mark.parametrize("mean", [0.4, 60.0], ids=["", "far-mean"])  # 60: the statistics take their second pass
@pytest.mark.parametrize("shape,groups,half,two", [
    ((2, 1280, 9, 7), 32, True, True), ((2, 1280, 9, 7), 32, False, True),     # rows of 63: pieces that a row's end cuts
    ((1, 1280, 21, 19), 32, True, True), ((1, 1280, 21, 19), 32, False, True),  # several slices, the last shorter
    ((3, 136, 7, 23), 17, True, True), ((3, 136, 7, 23), 17, False, True),     # 17 groups, a last tile of 8 channels
    ((2, 65, 8, 161), 65, True, True), ((2, 65, 10, 129), 65, False, False),   # a group per channel; no whole vectors
    ((1, 8, 300, 300), 1, True, True), ((1, 8, 300, 300), 1, False, True),     # one unit in 16 slices
    ((2, 320, 56, 48), 32, True, True), ((2, 320, 56, 48), 32, False, True),   # short runs, long units
    ((2, 320, 45, 56), 32, True, True), ((2, 320, 45, 56), 32, False, True),   # ... rows of no whole cache lines, 200 tiles a plane
    ((3, 320, 41, 56), 32, True, True), ((3, 320, 41, 56), 32, False, True),   # ... 180 tiles: no whole number per XCD
    ((1, 2560, 34, 32), 128, True, True),                                      # ... and more channels than positions
    ((20, 640, 2, 13), 32, False, False), ((40, 640, 2, 13), 32, False, True),  # units of 520: few of them, many
    ((40, 640, 2, 13), 32, True, True), ((60, 640, 1, 22), 32, False, False),   # planes much narrower than a tile
    ((16, 2560, 4, 4), 32, True, False), ((3, 136, 2, 5), 17, True, False)])   # short units
def test_groupnorm_tokens_in_two_launches(msd, orc, cuda, shape, groups, mean, half, two):
    """Statistics, then normalising tiles: against the oracle in 64 bits, eagerly and from graphs recorded on
    a stream without scratch, with a workspace (the same bits) and without (the kernels that need neither)."""
    import torch
    batch, channels, hw = shape[0], shape[1], int(np.prod(shape[2:]))
    x = orc.normal(shape, seed=sum(shape) + 5, sigma=1.5, mean=mean)
    g, b = _affine(orc, channels, 21)
    xin = orc.round_to_half(x) if half else x
    ref = orc.groupnorm64(xin, g, b, groups, 1e-6, False).astype(np.float32).reshape(batch, channels, hw).transpose(0, 2, 1)
    xd, gd, bd = _dev(xin, cuda, half), _dev(g, cuda), _dev(b, cuda)

    def check(got, what):
        (assert_close_f16 if half else assert_close_f32)(got.float().cpu().numpy(), ref, what=what)

    eager = msd.groupnorm_tokens(xd, gd, bd, groups, 1e-6)
    check(eager, "gn tokens, two launches")
    stream, lib = torch.cuda.Stream(), msd.load_library()
    assert _takes_two_launches(msd, xd, gd, bd, groups) == two
    assert lib.msd_release(stream.cuda_stream) == 0  # (an earlier stream may have had this handle)
    stream.wait_stream(torch.cuda.current_stream())
    # (the kernels that need no scratch do not split units: a unit that only fits in slices is left out)
    scratch_free = hw * channels // groups <= 20480
    with_workspace, without = torch.cuda.CUDAGraph(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(with_workspace, stream=stream):
        recorded = msd.groupnorm_tokens(xd, gd, bd, groups, 1e-6)
    plain = torch.empty_like(recorded)
    with torch.cuda.graph(without, stream=stream):
        assert not scratch_free or lib.msd_groupnorm_tokens(
            xd.data_ptr(), plain.data_ptr(), gd.data_ptr(), bd.data_ptr(), batch, channels, hw, groups, 1e-6,
            msd.DTYPE_F16 if half else msd.DTYPE_F32, stream.cuda_stream) == 0
    for _ in range(3):
        recorded.zero_()
        with_workspace.replay()
        torch.cuda.synchronize()
        assert torch.equal(recorded, eager)
        if scratch_free:
            plain.zero_()
            without.replay()
            torch.cuda.synchronize()
            check(plain, "gn tokens, recorded without scratch")


@pytest.mark.parametrize("shape,half", [((3, 320, 41, 56), True), ((3, 320, 41, 56), False), ((2, 1280, 9, 7), True), ((2, 65, 8, 161), True)])
def test_groupnorm_tokens_in_two_launches_on_other_xcd_counts(msd, orc, cuda, shape, half):
    """The tiles of planes whose rows are no whole cache lines are dealt out by XCD: every tile once, whatever their number."""
    import torch
    lib, groups = msd.load_library(), 65 if shape[1] == 65 else 32
    xd = torch.empty(shape, dtype=torch.float16 if half else torch.float32, device=cuda).normal_(0.4, 1.5)
    gd, bd = (_dev(t, cuda) for t in _affine(orc, shape[1], 26))
    assert _takes_two_launches(msd, xd, gd, bd, groups)
    want = msd.groupnorm_tokens(xd, gd, bd, groups, 1e-6)
    try:
        for xcds in (1, 2, 6, 16, 64):
            assert lib.msd_set_tuning(msd.TUNE_DEVICE_XCDS, xcds) == 0
            got = torch.full_like(want, float("nan"))
            assert lib.msd_groupnorm_tokens(
                xd.data_ptr(), got.data_ptr(), gd.data_ptr(), bd.data_ptr(), shape[0], shape[1], shape[2] * shape[3], groups, 1e-6,
                msd.DTYPE_F16 if half else msd.DTYPE_F32, torch.cuda.current_stream().cuda_stream) == 0
            assert torch.equal(got, want), xcds
    finally:
        assert lib.msd_set_tuning(msd.TUNE_DEVICE_XCDS, 0) == 0


@pytest.mark.parametrize("shape,half,two", [
    ((39, 1280, 16, 16), True, True), ((38, 1280, 16, 16), True, False),       # 24 MiB; more channels than positions
    ((20, 1280, 16, 16), False, True), ((24, 1280, 16, 16), False, False),     # a whole number of workgroups per CU
    ((16, 640, 36, 36), False, False),                                         # positions that leave a tile half empty
    ((48, 1280, 18, 18), True, False), ((18, 512, 24, 33), False, False),      # one launch that asks for gamma and beta behind the sums
    ((12, 640, 28, 28), False, False), ((40, 320, 20, 16), False, False)])     # (two writers); a small one that does not
def test_groupnorm_tokens_of_large_tensors(msd, orc, cuda, shape, half, two):
    import torch
    batch, channels, hw = shape[0], shape[1], shape[2] * shape[3]
    xd = torch.empty(shape, dtype=torch.float16 if half else torch.float32, device=cuda).normal_(0.4, 1.5)
    g, b = _affine(orc, channels, 24)
    gd, bd = _dev(g, cuda), _dev(b, cuda)
    assert _takes_two_launches(msd, xd, gd, bd, 32) == two
    got = msd.groupnorm_tokens(xd, gd, bd, 32, 1e-6)[::7].float().cpu().numpy()
    ref = orc.groupnorm64(xd[::7].float().cpu().numpy(), g, b, 32, 1e-6, False).astype(np.float32)
    ref = ref.reshape(-1, channels, hw).transpose(0, 2, 1)
    (assert_close_f16 if half else assert_close_f32)(got, ref, what="gn tokens, large")


def test_graphs_of_one_capture_stream_run_at_the_same_time(msd, orc, cuda):
    """Two graphs recorded on one stream, replayed on two: token norms in two launches, and norms in place of
    channels of no whole vectors, which outside a capture go through the stream's scratch."""
    import torch
    g, b = (_dev(t, cuda) for t in _affine(orc, 320, 23))
    capture = torch.cuda.Stream()
    graphs, inputs, wants, gots = [], [], [], []
    for i in range(2):
        x = torch.empty((2, 320, 64, 64), dtype=torch.float16, device=cuda).normal_(float(i), 1.0 + i)
        z = torch.empty((2, 320, 62, 66), dtype=torch.float16, device=cuda).normal_(float(2 * i), 1.0 + i)
        inputs.append((x, z))
        with torch.cuda.stream(capture):
            msd.init()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=capture):
            tokens = [msd.groupnorm_tokens(x, g, b, 32) for _ in range(20)]
            inplace = [z.clone() for _ in range(20)]
            for t in inplace:
                msd.groupnorm(t, g, b, 32, out=t)
        graph.replay()
        torch.cuda.synchronize()
        wants.append([t.clone() for t in tokens + inplace])
        gots.append(tokens + inplace)
        graphs.append(graph)
    streams = [torch.cuda.Stream() for _ in range(2)]
    for _ in range(5):
        for t in gots[0] + gots[1]:
            t.zero_()
        torch.cuda.synchronize()
        for graph, stream in zip(graphs, streams):
            with torch.cuda.stream(stream):
                graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(t, w) for i in range(2) for t, w in zip(gots[i], wants[i]))
    assert torch.equal(wants[0][0], wants[0][19]) and torch.equal(wants[0][20], wants[0][39])


def test_scratch_made_while_another_stream_is_captured(msd, orc, cuda):
    """Channels of no whole vectors on a stream that has no scratch yet, launched while another stream is being
    captured: the results are right, the capture is whole and no HIP error is left behind."""
    import ctypes

    import torch
    lib, hip = msd.load_library(), ctypes.CDLL("libamdhip64.so")
    shape = (2, 320, 62, 66)
    x = orc.round_to_half(orc.normal(shape, seed=77, sigma=1.5))
    g, b = _affine(orc, 320, 26)
    ref = orc.groupnorm64(x, g, b, 32, 1e-6, False).astype(np.float32).reshape(2, 320, -1)
    xd, zd, gd, bd = _dev(x, cuda, True), _dev(x, cuda, True), _dev(g, cuda), _dev(b, cuda)
    tokens = torch.empty((2, 62 * 66, 320), dtype=torch.float16, device=cuda)
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    assert lib.msd_release(stream.cuda_stream) == 0
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
        recorded = gd * 2
        assert lib.msd_groupnorm_tokens(xd.data_ptr(), tokens.data_ptr(), gd.data_ptr(), bd.data_ptr(), 2, 320, 62 * 66, 32,
                                        1e-6, msd.DTYPE_F16, stream.cuda_stream) == 0
        assert lib.msd_groupnorm(zd.data_ptr(), zd.data_ptr(), gd.data_ptr(), bd.data_ptr(), 2, 320, 62 * 66, 32, 1e-6, 0,
                                 msd.DTYPE_F16, stream.cuda_stream) == 0
        assert hip.hipPeekAtLastError() == 0
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(recorded, gd * 2)
    assert_close_f16(tokens.float().cpu().numpy(), ref.transpose(0, 2, 1), what="gn tokens, capture elsewhere")
    assert_close_f16(zd.float().cpu().numpy(), ref.reshape(shape), what="gn ragged, capture elsewhere")


def test_groupnorm_tokens_workspace_arguments(msd, cuda):
    import torch
    lib = msd.load_library()
    x, y = (torch.empty((2, 64, 16), dtype=torch.float16, device=cuda) for _ in range(2))
    w = torch.ones(64, device=cuda)
    ws = torch.empty(2 * 32 * msd.TOKENS_WORKSPACE_BYTES, dtype=torch.uint8, device=cuda)

    def call(workspace, size, groups=32):
        return lib.msd_groupnorm_tokens_workspace(x.data_ptr(), y.data_ptr(), w.data_ptr(), w.data_ptr(), 2, 64, 16, groups, 1e-6,
                                                  msd.DTYPE_F16, workspace, size, None)

    assert call(ws.data_ptr(), ws.numel()) == 0
    for bad in (call(None, ws.numel()), call(ws.data_ptr(), ws.numel() - 1), call(ws.data_ptr() + 4, ws.numel()),
                call(x.data_ptr(), ws.numel()), call(y.data_ptr(), ws.numel()), call(ws.data_ptr(), ws.numel(), 0)):
        assert bad == 1
    assert msd.status() == 0


@pytest.mark.parametrize("halves", [(True, True), (True, False), (False, False)], ids=["f16", "f16-f32", "f32"])
def test_groupnorm_tokens_from_two_threads_on_one_stream(msd, orc, cuda, halves):
    """The two launches of a call stay together when another thread launches on the same stream, with
    elements of its own type or of the other."""
    import threading

    import torch
    g, b = (_dev(t, cuda) for t in _affine(orc, 320, 22))
    xs = [torch.empty((2, 320, 64, 64), dtype=torch.float16 if half else torch.float32, device=cuda)
          .normal_(float(i), 1.0 + i) for i, half in enumerate(halves)]
    want = [msd.groupnorm_tokens(x, g, b, 32) for x in xs]
    got, start = [[], []], threading.Barrier(2)

    def work(i):
        start.wait()
        for _ in range(100):
            got[i].append(msd.groupnorm_tokens(xs[i], g, b, 32))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(len(got[i]) == 100 and all(torch.equal(o, want[i]) for o in got[i]) for i in range(2))


@pytest.mark.parametrize("half", [False, True], ids=["f32", "f16"])
@pytest.mark.parametrize("shape", [(2, 320, 4096), (2, 4096, 320), (1, 1280, 64), (3, 100, 36), (2, 7, 5),
                                   (1, 64, 64), (5, 68, 132), (1, 1, 8),
                                   # 16-byte pieces on both sides with ragged tiles, one tile, thin planes
                                   (3, 72, 200), (2, 8, 8), (1, 136, 64), (2, 16, 1000), (4, 264, 24)])
def test_permute_0_2_1(msd, orc, cuda, shape, half):
    import torch
    x = orc.normal(shape, seed=sum(shape))
    xin = orc.round_to_half(x) if half else x
    got = msd.permute_0_2_1(_dev(xin, cuda, half))
    assert np.array_equal(got.float().cpu().numpy(), orc.permute_0_2_1(xin))
    assert torch.equal(msd.permute_0_2_1(got), _dev(xin, cuda, half))  # its own inverse


@pytest.mark.parametrize("half", [False, True], ids=["f32", "f16"])
@pytest.mark.parametrize("shape", [(2, 63, 1280), (2, 1280, 63), (1, 65, 127), (3, 1, 9), (2, 9, 1), (1, 130, 66),
                                   (4, 63, 1280), (4, 1280, 63), (24, 65, 127), (23, 130, 66), (1, 5, 40000), (1, 40000, 7),
                                   (33, 65, 127), (31, 130, 66), (23, 65, 127),
                                   (700, 17, 17), (650, 20, 17), (3000, 3, 64)])   # tiles; planes that fill too few of them
def test_permute_0_2_1_ragged_and_unaligned(msd, orc, cuda, shape, half):
    """Rows that start at any element and end inside a 16-byte piece, in tensors that start one
    element past an aligned address, with nothing written around the output."""
    import torch
    n = int(np.prod(shape))
    x = orc.normal(shape, seed=sum(shape))
    x = orc.round_to_half(x) if half else x
    src = torch.zeros(n + 2, dtype=torch.float16 if half else torch.float32, device=cuda)
    src[1:n + 1] = _dev(x, cuda, half).reshape(-1)
    dst = torch.full_like(src, 7.0)
    elt = src.element_size()
    assert msd.load_library().msd_permute_0_2_1(src.data_ptr() + elt, dst.data_ptr() + elt, *shape,
                                                msd.DTYPE_F16 if half else msd.DTYPE_F32, None) == 0
    torch.cuda.synchronize()
    got = dst.float().cpu().numpy()
    assert np.array_equal(got[1:n + 1], orc.permute_0_2_1(x).reshape(-1))
    assert got[0] == 7.0 and got[n + 1] == 7.0


@pytest.mark.parametrize("shape", [(3, 4, 12), (300, 12, 4), (2, 20, 36), (1, 68, 132), (2, 252, 1280), (2, 1280, 252)])
def test_permute_0_2_1_in_halves_of_a_piece(msd, orc, cuda, shape):
    """2-byte sides in multiples of four, and of eight in planes that start in the middle of a piece."""
    import torch
    for scale, offset in ((1, 0), (1, 4), (2, 4)):
        i, j, k = shape[0], shape[1] * scale, shape[2] * scale
        n = i * j * k
        x = orc.round_to_half(orc.normal((i, j, k), seed=sum(shape) + scale))
        src = torch.zeros(n + 16, dtype=torch.float16, device=cuda)
        src[offset:n + offset] = _dev(x, cuda, True).reshape(-1)
        dst = torch.full_like(src, 7.0)
        assert msd.load_library().msd_permute_0_2_1(src.data_ptr() + 2 * offset, dst.data_ptr() + 2 * offset, i, j, k,
                                                    msd.DTYPE_F16, None) == 0
        torch.cuda.synchronize()
        got = dst.float().cpu().numpy()
        assert np.array_equal(got[offset:n + offset], orc.permute_0_2_1(x).reshape(-1))
        assert (got[:offset] == 7.0).all() and (got[n + offset:] == 7.0).all()


def test_permute_0_2_1_of_a_row_beyond_the_tiles_of_a_grid(msd, cuda):
    """The first length whose tiles of 256 lanes are 2^32 lanes, which no launch takes."""
    import torch
    j, k = 5, 2 ** 30 - 63
    x = torch.randint(-2 ** 15, 2 ** 15, (1, j, k), dtype=torch.int16, device=cuda)
    got = msd.permute_0_2_1(x.view(torch.float16)).view(torch.int16)
    assert got.shape == (1, k, j) and all(torch.equal(got[0, :, i], x[0, i]) for i in range(j))


def test_fused_argument_checks(msd, cuda):
    lib = msd.load_library()
    assert lib.msd_chunk_add_groupnorm(None, None, None, None, None, 1, 32, 16, 32, 1e-5, 0, 0, None) == 1
    assert lib.msd_add_layernorm(None, None, None, None, None, None, 4, 64, 1e-5, 0, None) == 1
    assert lib.msd_chunkwise_add(None, None, None, 16, 0, 0, None) == 1
    assert lib.msd_elemwise_add(None, None, None, 0, 0, None) == 0
    import torch
    x = torch.zeros(32 * 64, device=cuda)
    p = ctypes.c_void_p(x.data_ptr())
    assert lib.msd_groupnorm_tokens(p, p, p, p, 1, 32, 64, 32, 1e-6, 0, None) == 1  # y must not be x


@pytest.mark.parametrize("half", [False, True], ids=["f32", "f16"])
@pytest.mark.parametrize("extra", [-1, 0, 1, 65])
@pytest.mark.parametrize("waves", [22, 48])
def test_elementwise_launches_around_a_full_chip(msd, cuda, waves, extra, half):
    """Vectors on both sides of 22 and 48 wavefronts per CU (256 CUs), from where on a workgroup is one wavefront, with elements
    left over: the bits of short launches."""
    import torch
    dtype, epv = (torch.float16, 8) if half else (torch.float32, 4)
    vecs, left = waves * 64 * 256 + extra, epv - 1
    g = torch.Generator(device=cuda).manual_seed(extra + 7)
    x, y = (torch.randn(vecs * epv + left, device=cuda, generator=g).to(dtype) for _ in range(2))
    for op in (msd.silu, msd.gelu, msd.quick_gelu):
        got = op(x)
        for a, b in ((0, 4096), (x.numel() // 2 // 64 * 64, x.numel() // 2 // 64 * 64 + 4096), (x.numel() // 64 * 64 - 4096, x.numel())):
            assert torch.equal(got[a:b], op(x[a:b].clone()))
    whole = slice(0, vecs * epv)
    assert torch.equal(msd.elemwise_add(x[whole], y[whole]), x[whole] + y[whole])
    assert torch.equal(msd.elemwise_add(x, y), x + y)
    chunk = vecs * epv // 4 if vecs % 4 == 0 else vecs * epv  # (whole vectors per chunk)
    addend = torch.randn(vecs * epv // chunk, device=cuda, generator=g).to(dtype)
    assert torch.equal(msd.chunkwise_add(x[whole], addend, chunk), (x[whole].view(-1, chunk) + addend[:, None]).view(-1))
