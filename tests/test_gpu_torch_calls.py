"""The package's calls in native code (csrc/torch_calls.cpp) against their general path: the same bits, the same outputs,
the same refusals."""
import threading

import pytest

pytestmark = pytest.mark.gpu


class _General:
    """Stands for native calls that find no call plain."""

    def __getattr__(self, name):
        return lambda *args: None


def _cases(torch, msd, cuda, half):
    g = torch.Generator(device=cuda).manual_seed(5)
    dtype = torch.float16 if half else torch.float32

    def rnd(*shape):
        return torch.randn(shape, device=cuda, generator=g).to(dtype)

    x, rows, emb = rnd(2, 64, 8, 6), rnd(6, 64), rnd(2, 64)
    gamma, beta = torch.randn(64, device=cuda, generator=g), torch.randn(64, device=cuda, generator=g)
    ws, bs = [rnd(n, 64) for n in (3, 40, 1)], [torch.randn(3, device=cuda, generator=g), None, torch.randn(1, device=cuda, generator=g)]
    steps = torch.tensor([981, 1], device=cuda)
    e = msd.ACT_SILU
    return {
        "groupnorm": [(x, gamma, beta, 32), (x, gamma, beta, 8, 1e-3, True), (x, gamma, beta, 8, 1e-3, False, torch.empty_like(x)),
                      (x, gamma, beta, 8, 1e-3, False, None, True), (x, gamma, beta, 7), (x, gamma[:63], beta, 8),
                      (x, gamma.half(), beta, 8), (x.cpu(), gamma, beta, 8), (x, gamma, beta.cpu(), 8), (x.transpose(2, 3), gamma, beta, 8),
                      (x, gamma, beta, 8, 1e-3, False, torch.empty_like(x)[:1]), (x, gamma, beta, 8, 1e-3, False, x.flatten()),
                      (x, gamma, beta, -1), (x, gamma, beta, 2.0), (x.double(), gamma, beta, 8), (x, gamma, beta, 8, 1e-3, 1),
                      (x[0, 0, 0], gamma, beta, 8), (x[:0], gamma, beta, 8), (x, None, beta, 8), (x, torch.nn.Parameter(gamma), beta, 8)],
        "chunk_add_groupnorm": [(x, emb, gamma, beta, 8), (x, emb[:1], gamma, beta, 8), (x, emb, gamma, beta, 8, 1e-5, True, x.clone()),
                                (x, x.view(-1)[:128].view(2, 64), gamma, beta, 8, 1e-5, True, x)],  # (an addend in the output)
        "groupnorm_tokens": [(x, gamma, beta, 8), (x, gamma, beta, 8, 1e-2), (x, gamma, beta, 7), (x.cpu(), gamma, beta, 8)],
        "permute_0_2_1": [(x.view(2, 64, 48),), (x,), (x.view(2, 64, 48).transpose(1, 2),), (rows[:0].view(0, 8, 8),)],
        "layernorm": [(rows, gamma, beta), (rows, gamma, beta, 1e-2, torch.empty_like(rows)), (rows, gamma, beta[:8]), (rows[:, ::2], gamma, beta),
                      (rows, gamma, beta, None), (rows.view(-1)[1:65], gamma, beta)],
        "add_layernorm": [(rows, rows, gamma, beta), (rows, emb, gamma, beta), (rows.clone(), rows, gamma, beta, 1e-2, torch.empty_like(rows), None)],
        "elemwise_add": [(rows, rows), (rows, emb), (rows, rows, torch.empty_like(rows)), (rows, rows.cpu()), (rows, 1.0)],
        "chunkwise_add": [(x, emb, 48), (x, emb, 47), (x, emb, 0), (x, emb, 48, torch.empty_like(x)), (x, rows, 48)],
        "geglu": [(rows,), (rows, rnd(6, 32)), (rows, rnd(6, 31)), (rnd(3, 7),), (rnd(2, 3, 16),)],
        "silu": [(rows,), (rows, torch.empty_like(rows)), (rows.to(torch.bfloat16),)], "gelu": [(rows,), (rows, emb)], "quick_gelu": [(x,)],
        "timestep_embedding": [(steps, 320), (steps, 320, 10000.0, dtype), (steps, 321), (steps, 320, 1e4, torch.float64), (steps.cpu(), 320),
                               (steps, 16, -1.0)],
        "linear_rows": [(rows, ws[1]), (rows, ws[1], None, e, e), (rows, ws[0], bs[0], 0, 0, rnd(6, 3)), (rows, ws[0], bs[0], 0, 0, rnd(6, 4)),
                        (rows, ws[0], bs[2]), (rows, ws[0].to(torch.float64)), (rows, rnd(4, 63)), (rnd(9, 64), ws[0]), (rows, ws[0], None, 3), (x, ws[0])],
        "linear_rows_grouped": [(emb, ws), (emb, ws, bs, e), (emb, tuple(ws), bs), (emb, ws, bs[:1]), (emb, [ws[0], rows[:, :8]]), (emb, []),
                                (rnd(9, 64), ws), (emb, ws, [None] * 4, 0, e)],
        "softmax": [(rows,), (rows, True), (rows, 1), (rows, False, rows.clone()), (rows, False, emb), (rows.t(),)],
        "ddim_update": [(rows, rows * 0.5, 0.5, 0.6, 0.7), (rows, rows, 0.5, 0.6, 0.7, torch.empty_like(rows)), (rows, rows, 0.0, 0.6, 0.7),
                        (rows, emb, 0.5, 0.6, 0.7), (rows, rows, "a", 0.6, 0.7)],
    }


def _outcome(torch, f, args):
    """What the call returns and leaves in its tensors, or how it is refused."""
    try:
        got = f(*args)
    except Exception as e:  # (TypeError, MsdError, ctypes.ArgumentError, ...)
        return type(e).__name__, str(e)
    flat = list(got) if isinstance(got, (list, tuple)) else [got]
    return [type(got).__name__] + [(t.clone(), next((i for i, a in enumerate(args) if a is t), None)) for t in flat]


@pytest.mark.parametrize("half", [False, True], ids=["f32", "f16"])
def test_native_calls_are_the_general_ones(msd, cuda, half, monkeypatch):
    import torch
    twice = _cases(torch, msd, cuda, half), _cases(torch, msd, cuda, half)  # (some calls write into what later ones read)
    for name, cases in twice[0].items():
        f = getattr(msd, name)
        for i, args in enumerate(cases):
            native = _outcome(torch, f, args)
            with monkeypatch.context() as m:
                m.setattr(msd, "_native", _General())
                general = _outcome(torch, f, twice[1][name][i])
            what = "%s, call %d" % (name, i)
            assert len(native) == len(general) and native[0] == general[0], what
            for a, b in zip(native[1:], general[1:]):
                if isinstance(a, tuple):
                    assert a[1] == b[1] and a[0].dtype == b[0].dtype and a[0].shape == b[0].shape, what
                    assert torch.equal(a[0].nan_to_num(7.0), b[0].nan_to_num(7.0)), what
                else:
                    assert a == b, what


def test_native_calls_take_the_plain_call_and_leave_the_others(msd, cuda):
    import torch
    x, g, b = torch.randn(4, 64, device=cuda), torch.ones(64, device=cuda), torch.zeros(64, device=cuda)
    native = msd._bind_native()
    assert torch.equal(native.layernorm(x, g, b, 1e-5, None), msd.layernorm(x, g, b))

    class Sub(torch.Tensor):
        pass

    assert native.layernorm(x.as_subclass(Sub), g, b, 1e-5, None) is None
    assert type(msd.layernorm(x.as_subclass(Sub), g, b)) is Sub
    assert native.layernorm(x, g, b, 1e-5) is None and native.silu() is None  # (the package passes all arguments)
    with torch.device(cuda):  # a mode that functions of torch's go through
        assert native.layernorm(x, g, b, 1e-5, None) is None
        under_mode = msd.layernorm(x, g, b)
    assert torch.equal(under_mode, msd.layernorm(x, g, b))
    seen = []

    def row(v):
        seen.append(native.silu(v, None))
        return v * 2

    torch.vmap(row)(x)
    assert seen == [None]
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    image = torch.randn(2, 64, 8, 8, device=cuda)
    with torch.cuda.graph(graph, stream=stream):  # a recorded token norm brings a workspace
        assert native.groupnorm_tokens(image, g, b, 8, 1e-6) is None
        recorded = msd.layernorm(x, g, b)
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(recorded, msd.layernorm(x, g, b))


def test_new_outputs_have_the_strides_of_the_general_path(msd, cuda, monkeypatch):
    """torch.empty_like keeps the strides of axes of length one, which a contiguous tensor may have any of."""
    import torch
    gamma, beta = torch.ones(64, device=cuda), torch.zeros(64, device=cuda)
    planes = torch.randn(2, 64, 1, 1, device=cuda).to(memory_format=torch.channels_last)
    one = torch.randn(3, 5, 64, device=cuda)[:1, 2:3]
    none = torch.randn(2, 64, 3, 0, device=cuda).to(memory_format=torch.channels_last)
    odd = [planes, one, torch.randn(4, 64, device=cuda).as_strided((1, 64), (7, 1)), none, torch.randn(2, 64, 1, 8, device=cuda)]
    assert planes.is_contiguous() and planes.stride(1) == 1 and one.is_contiguous() and one.stride(0) == 320
    calls = [(msd.silu, x) for x in odd] + [(msd.gelu, x) for x in odd] + [(lambda x: msd.elemwise_add(x, x), x) for x in odd] + \
        [(lambda x: msd.groupnorm(x, gamma, beta, 8), planes), (lambda x: msd.groupnorm(x, gamma, beta, 8), odd[-1]),
         (lambda x: msd.layernorm(x, gamma, beta), one), (lambda x: msd.add_layernorm(x, x, gamma, beta)[1], one),
         (lambda x: msd.chunk_add_groupnorm(x, x, gamma, beta, 8), planes), (msd.softmax, one),
         (lambda x: msd.ddim_update(x, x, 0.5, 0.6, 0.7), one), (lambda x: msd.chunkwise_add(x, x, 1), planes)]
    for i, (f, x) in enumerate(calls):
        native = f(x)
        with monkeypatch.context() as m:
            m.setattr(msd, "_native", _General())
            general = f(x)
        assert native.stride() == general.stride() == torch.empty_like(x).stride(), i
        assert torch.equal(native, general), i


def test_native_calls_use_the_threads_stream(msd, cuda):
    """Threads on streams of their own: what a call reads was written on its stream just before."""
    import torch
    wrong = []

    def work(i):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for k in range(40):
                x = torch.full((64, 256), float(i + k), device=cuda)
                y = msd.elemwise_add(x, x)
                if not bool((y == 2.0 * (i + k)).all()):
                    wrong.append((i, k))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not wrong


# Which calls of _cases are plain: the extension makes them, or refuses them with the library's code, and leaves the others.
_PLAIN = {
    "groupnorm": {0, 1, 2, 3, 4, 11, 17, 19}, "chunk_add_groupnorm": {0, 2, 3}, "groupnorm_tokens": {0, 1, 2},
    "permute_0_2_1": {0, 3}, "layernorm": {0, 1, 5}, "add_layernorm": {0, 2}, "elemwise_add": {0, 2}, "chunkwise_add": {0, 3},
    "geglu": {0, 1, 3, 4}, "silu": {0, 1}, "gelu": {0}, "quick_gelu": {0}, "timestep_embedding": {0, 1, 2, 5},
    "linear_rows": {0, 1, 2, 7, 8}, "linear_rows_grouped": {0, 1, 5, 6, 7}, "softmax": {0, 1, 3}, "ddim_update": {0, 1, 2},
}


class _Recorder:
    """Passes calls on to the extension and notes whether it made them."""

    def __init__(self, native):
        self.native, self.made = native, []

    def __getattr__(self, name):
        def call(*args):
            self.made.append((name, True))  # (so it stands if the extension raises)
            done = getattr(self.native, name)(*args)
            self.made[-1] = name, done is not None
            return done
        return call


@pytest.mark.parametrize("half", [False, True], ids=["f32", "f16"])
def test_every_plain_call_is_made_by_the_extension_and_no_other(msd, cuda, half, monkeypatch):
    import torch
    cases = _cases(torch, msd, cuda, half)
    native = msd._bind_native()
    entries = {n for n in dir(native) if not n.startswith("__")} - {"bind", "names", "built_for"}
    assert set(cases) == set(_PLAIN) == entries
    recorder = _Recorder(native)
    monkeypatch.setattr(msd, "_native", recorder)
    for name, calls in cases.items():
        for i, args in enumerate(calls):
            recorder.made.clear()
            _outcome(torch, getattr(msd, name), args)
            assert (name, True) in recorder.made if i in _PLAIN[name] else recorder.made in ([], [(name, False)]), (name, i)


def test_native_calls_wait_for_what_is_on_the_threads_stream(msd, cuda):
    """The operand is written behind work that takes far longer than the host needs to reach the call's launch: on any other
    stream the call would read what was there before."""
    import torch
    wrong = []

    def work(i):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            big, x = torch.empty(1 << 28, device=cuda), torch.full((64, 256), -1.0, device=cuda)  # (1 GiB)
            for k in range(4):
                x.fill_(-1.0)
                stream.synchronize()
                for _ in range(16):  # (some 3 ms)
                    big.fill_(float(k))
                x.fill_(float(i + k))
                waits = not stream.query()
                y = msd.elemwise_add(x, x)
                if not waits or not bool((y == 2.0 * (i + k)).all()):
                    wrong.append((i, k, waits))

    for i in range(4):  # one after the other: threads that wait for the interpreter could let the work end before the call
        thread = threading.Thread(target=work, args=(i,))
        thread.start()
        thread.join()
    assert not wrong
