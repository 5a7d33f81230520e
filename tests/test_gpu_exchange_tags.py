"""Launches of cut units one after the other on one scratch, a stream's or the fixed one, in changing numbers of slices
(csrc/groupnorm.hip: gn_exchange): every launch finds its slices agreed on the tag, so none of them gives up waiting, and each
result is that of the first launch with its number of slices, bit for bit, eagerly and from a replayed graph.  The tokens'
kernel shares the words."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SPLITS = [2, 64, 4, 8, 2, 16, 32, 4, 64, 2]


@pytest.mark.parametrize("batch,channels,side", [(1, 320, 64), (2, 64, 64)])
@pytest.mark.parametrize("half", [False, True], ids=["f32", "f16"])
def test_launches_in_changing_slices_agree_on_the_tag(msd, orc, cuda, half, batch, channels, side):
    import torch
    lib = msd.load_library()
    x = torch.from_numpy(orc.normal((batch, channels, side, side), seed=channels, sigma=2.0)).to(cuda)
    x = x.half() if half else x
    gamma, beta = (torch.from_numpy(orc.normal((channels,), seed=s)).to(cuda) for s in (1, 2))
    out = [torch.empty_like(x) for _ in SPLITS]

    def launches():
        for split, y in zip(SPLITS, out):
            torch.add(x, 0, out=y)
            assert lib.msd_set_tuning(msd.TUNE_GN_SPLIT, split) == 0
            msd.groupnorm(y, gamma, beta, 32, 1e-5, True, out=y)

    try:
        assert lib.msd_set_tuning(msd.TUNE_GN_WRITERS, 1) == 0
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            msd.init()
            msd.gn_fallbacks(reset=True)
            launches()
            assert lib.msd_set_tuning(msd.TUNE_GN_SPLIT, 4) == 0
            tokens = msd.groupnorm_tokens(x, gamma, beta, 32, 1e-5)
            first = [y.clone() for y in out]
            launches()
        torch.cuda.synchronize()
        of = {}
        for split, a, b in zip(SPLITS, first, out):
            assert torch.equal(a, b) and torch.equal(of.setdefault(split, a), a), split
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            launches()
        assert lib.msd_set_tuning(msd.TUNE_GN_SPLIT, 4) == 0
        for _ in range(3):
            for y in out:
                y.zero_()
            torch.cuda.synchronize()
            with torch.cuda.stream(stream):
                graph.replay()
                launches_between = msd.groupnorm_tokens(x, gamma, beta, 32, 1e-5)
            torch.cuda.synchronize()
            assert all(torch.equal(a, b) for a, b in zip(first, out)) and torch.equal(tokens, launches_between)
        with torch.cuda.stream(stream):
            assert msd.gn_fallbacks() == 0
    finally:
        lib.msd_set_tuning(msd.TUNE_GN_SPLIT, 0)
        lib.msd_set_tuning(msd.TUNE_GN_WRITERS, 0)
    # against the oracle, within what another order of the sums gives (tests of the kernel itself: test_gpu_parity.py)
    xin = x.float().cpu().numpy()
    ref = orc.groupnorm(xin, gamma.cpu().numpy(), beta.cpu().numpy(), 32, 1e-5, silu=True)
    got = first[0].float().cpu().numpy()
    bound = (2.0 ** -10 if half else 0.0) * np.abs(ref) + 1e-5 * np.maximum(1.0, np.abs(ref))  # a last bit of fp16, and 1e-5
    assert np.all(np.abs(got - ref) <= bound)


@pytest.mark.parametrize("half", [False, True], ids=["f32", "f16"])
def test_fixed_scratch_in_changing_slices_from_two_streams_in_turn(msd, orc, cuda, half):
    """msd_groupnorm_noalloc in place, calls on two streams that events put in order, units of two tensors in changing numbers
    of slices on the one array of the device: the bits of the same launches on a stream's own scratch, and nobody gives up."""
    import torch
    lib, code, vp = msd.load_library(), msd.DTYPE_F16 if half else msd.DTYPE_F32, ctypes.c_void_p
    shapes = [(1, 320, 4096), (2, 64, 4096)]
    xs = [torch.from_numpy(orc.normal(s, seed=s[1] + 1, sigma=2.0)).to(cuda) for s in shapes]
    xs = [x.half() if half else x for x in xs]
    affine = [[torch.from_numpy(orc.normal((s[1],), seed=seed)).to(cuda) for seed in (3, 4)] for s in shapes]

    def call(fn, i, y, stream):
        (batch, channels, hw), (g, b) = shapes[i], affine[i]
        assert fn(vp(y.data_ptr()), vp(y.data_ptr()), vp(g.data_ptr()), vp(b.data_ptr()), batch, channels, hw, 32, 1e-5, 1, code,
                  vp(stream.cuda_stream)) == 0

    streams = [torch.cuda.Stream() for _ in range(2)]
    msd.init()
    msd.gn_fallbacks(reset=True)
    try:
        assert lib.msd_set_tuning(msd.TUNE_GN_WRITERS, 1) == 0
        for round_ in range(3):
            for turn, split in enumerate(SPLITS):
                assert lib.msd_set_tuning(msd.TUNE_GN_SPLIT, split) == 0
                i, stream = (turn + round_) % 2, streams[turn % 2]
                stream.wait_stream(torch.cuda.current_stream())
                stream.wait_stream(streams[(turn + 1) % 2])
                with torch.cuda.stream(stream):
                    got = xs[i].clone()
                    call(lib.msd_groupnorm_noalloc, i, got, stream)
                torch.cuda.current_stream().wait_stream(stream)
                want = xs[i].clone()
                call(lib.msd_groupnorm, i, want, torch.cuda.current_stream())
                torch.cuda.synchronize()
                assert torch.equal(got, want), (round_, split)
        assert msd.gn_fallbacks() == 0
    finally:
        lib.msd_set_tuning(msd.TUNE_GN_SPLIT, 0)
        lib.msd_set_tuning(msd.TUNE_GN_WRITERS, 0)
