"""ctypes access to the MI355X norm / activation / embedding library.

The product is the native code under csrc/ (HIP kernels behind the C ABI of
include/msd_hip.h, and the C++ layer objects on top of it).  This module only
loads the built libraries and passes torch tensors' device pointers and the
current torch stream through the C ABI; torch is used for device memory and
streams, nothing else.  There is no fallback: if the library was not built
the loader raises.
"""
import ctypes
import importlib.util
import os
import sys
import warnings

_PKG_DIR = os.path.dirname(os.path.abspath(__file__))
CSRC_DIR = os.path.join(_PKG_DIR, "csrc")
LIB_HIP_PATH = os.path.join(CSRC_DIR, "libmsd_hip.so")
LIB_NN_PATH = os.path.join(CSRC_DIR, "libmsd_nn.so")
TORCH_CALLS_PATH = os.path.join(CSRC_DIR, "msd_torch_calls.so")

DTYPE_F32 = 0
DTYPE_F16 = 1
TUNE_GN_SPLIT, TUNE_GN_THREADS, TUNE_LN_CHUNK, TUNE_LN_THREADS, TUNE_GEGLU_VECTORS, TUNE_ACT_VECTORS, \
    TUNE_SOFTMAX_ROWS, TUNE_GN_SPIN_LIMIT, TUNE_GN_WRITERS, TUNE_DEVICE_CUS, TUNE_DEVICE_XCDS, \
    TUNE_GN_PLAN_RULE_ONLY = range(12)
ERR_SCRATCH_LIMIT = -2
TOKENS_WORKSPACE_BYTES = 128  # per (sample, group): MSD_TOKENS_WORKSPACE_BYTES of include/msd_hip.h

# every symbol include/msd_hip.h declares
C_ABI_SYMBOLS = (
    "msd_version", "msd_error_string", "msd_init", "msd_release", "msd_shutdown", "msd_status",
    "msd_gn_fallbacks", "msd_set_tuning", "msd_groupnorm", "msd_groupnorm_noalloc", "msd_groupnorm_plan", "msd_layernorm", "msd_geglu",
    "msd_silu", "msd_gelu", "msd_quick_gelu", "msd_timestep_embedding", "msd_ddim_timesteps",
    "msd_elemwise_add", "msd_chunkwise_add", "msd_chunk_add_groupnorm", "msd_add_layernorm", "msd_copy",
    "msd_groupnorm_tokens", "msd_groupnorm_tokens_workspace", "msd_permute_0_2_1",
    "msd_linear_rows", "msd_linear_rows_grouped", "msd_softmax", "msd_alphas_cumprod", "msd_ddim_schedule", "msd_ddim_update",
)
ACT_NONE, ACT_SILU = 0, 1

_lib = None


class MsdError(RuntimeError):
    pass


def load_library(path=None):
    """Loads libmsd_hip.so (built in-tree) and declares the C ABI signatures."""
    global _lib
    if _lib is not None and path is None:
        return _lib
    path = path or LIB_HIP_PATH
    if not os.path.exists(path):
        raise MsdError(
            "native library %s is missing: build it with `python -c 'import __graft_entry__ as g;"
            " g.build()'` (there is no non-native fallback)" % path)
    lib = ctypes.CDLL(path, mode=ctypes.RTLD_GLOBAL)
    vp, sz, fl, it = ctypes.c_void_p, ctypes.c_size_t, ctypes.c_float, ctypes.c_int
    lib.msd_version.restype = it
    lib.msd_error_string.restype = ctypes.c_char_p
    lib.msd_error_string.argtypes = [it]
    lib.msd_init.argtypes = [vp]
    lib.msd_shutdown.argtypes = []
    lib.msd_status.argtypes = [vp]
    lib.msd_release.argtypes = [vp]
    lib.msd_gn_fallbacks.argtypes = [vp, ctypes.POINTER(ctypes.c_uint), it]
    lib.msd_set_tuning.argtypes = [it, it]
    lib.msd_groupnorm.argtypes = [vp, vp, vp, vp, sz, sz, sz, sz, fl, it, it, vp]
    lib.msd_groupnorm_noalloc.argtypes = [vp, vp, vp, vp, sz, sz, sz, sz, fl, it, it, vp]
    lib.msd_groupnorm_plan.argtypes = [sz, sz, sz, sz, it, it, it] + [ctypes.POINTER(ctypes.c_int)] * 4
    lib.msd_layernorm.argtypes = [vp, vp, vp, vp, sz, sz, fl, it, vp]
    lib.msd_geglu.argtypes = [vp, vp, sz, sz, it, vp]
    lib.msd_copy.argtypes = [vp, vp, sz, vp]
    lib.msd_permute_0_2_1.argtypes = [vp, vp, sz, sz, sz, it, vp]
    lib.msd_groupnorm_tokens.argtypes = [vp, vp, vp, vp, sz, sz, sz, sz, fl, it, vp]
    lib.msd_groupnorm_tokens_workspace.argtypes = [vp, vp, vp, vp, sz, sz, sz, sz, fl, it, vp, sz, vp]
    lib.msd_elemwise_add.argtypes = [vp, vp, vp, sz, it, vp]
    lib.msd_chunkwise_add.argtypes = [vp, vp, vp, sz, sz, it, vp]
    lib.msd_chunk_add_groupnorm.argtypes = [vp, vp, vp, vp, vp, sz, sz, sz, sz, fl, it, it, vp]
    lib.msd_add_layernorm.argtypes = [vp, vp, vp, vp, vp, vp, sz, sz, fl, it, vp]
    for name in ("msd_silu", "msd_gelu", "msd_quick_gelu"):
        getattr(lib, name).argtypes = [vp, vp, sz, it, vp]
    lib.msd_timestep_embedding.argtypes = [vp, vp, sz, sz, fl, it, vp]
    lib.msd_ddim_timesteps.argtypes = [it, ctypes.POINTER(ctypes.c_int), it]
    lib.msd_linear_rows.argtypes = [vp, vp, vp, vp, sz, sz, sz, it, it, it, vp]
    lib.msd_softmax.argtypes = [vp, vp, sz, sz, it, it, vp]
    lib.msd_linear_rows_grouped.argtypes = [vp, ctypes.POINTER(vp), ctypes.POINTER(vp), ctypes.POINTER(vp),
                                            ctypes.POINTER(sz), sz, sz, sz, it, it, it, vp]
    flp, inp = ctypes.POINTER(ctypes.c_float), ctypes.POINTER(ctypes.c_int)
    lib.msd_alphas_cumprod.argtypes = [flp]
    lib.msd_ddim_schedule.argtypes = [it, inp, flp, flp, flp, it]
    lib.msd_ddim_update.argtypes = [vp, vp, vp, sz, fl, fl, fl, it, vp]
    for name in C_ABI_SYMBOLS:
        if name != "msd_error_string":
            getattr(lib, name).restype = it
    _lib = lib
    if not isinstance(_native, _Unbound):
        _bind_addresses(_native)
    return lib


def check(code):
    if code != 0:
        raise MsdError("msd call failed with code %d: %s"
                       % (code, load_library().msd_error_string(code).decode()))


# What a call does on the host is most of a small call's time (a LayerNorm of 154 rows: a kernel of 2.2 us behind 2.5 to
# 3.5 us of the runtime's launch), so plain calls (dense device tensors that fit each other, no mode or transform around
# them) go through csrc/torch_calls.cpp, which checks them, makes the outputs and calls the C ABI; it returns None for any
# other, which the general path below it then makes or refuses.  Eager passes, us, from Python and so: four calls of a
# sampler's tick 25.0 -> 14.4, the 49 of a text encoder 325 -> 198 (to 222), 22 grouped projections 53 -> 15.3, the 8 of a
# 640-channel transformer block 55.6 -> 35.8.
class _Unbound:
    """Stands for the native calls until the first one."""

    def __getattr__(self, name):
        return getattr(_bind_native(), name)


class _NoNative:
    """Stands for the native calls where there are none: every call takes its general path."""

    def __getattr__(self, name):
        return lambda *args: None

    def names(self):
        return []

    def bind(self, addresses, check):
        pass


_native = _Unbound()


def _bind_addresses(native):
    native.bind({name: ctypes.cast(getattr(_lib, name), ctypes.c_void_p).value for name in native.names()}, check)


def _running(torch):
    """The Python and the torch at hand, as build.py names those that the extension is compiled for."""
    return "Python %d.%d, torch %s (%s)" % (sys.version_info[:2] + (torch.version.__version__, torch.version.git_version))


def _load_native(torch):
    """The extension, or what stands for it where it is not built or was built for another torch: the C ABI takes tensors of
    any torch, but the extension reads them as its own torch lays them out."""
    spec = importlib.util.spec_from_file_location("msd_torch_calls", TORCH_CALLS_PATH)
    try:
        native = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(native)
        built_for = getattr(native, "built_for", "another torch")
        if built_for == _running(torch):
            return native
        why = "was built for %s, this is %s" % (built_for, _running(torch))
    except ImportError as e:  # (no such file, or symbols that this torch does not have)
        why = "does not load: %s" % e
    warnings.warn("%s %s; a call takes about 2.5 us longer without it (run __graft_entry__.build())" % (TORCH_CALLS_PATH, why),
                  RuntimeWarning, stacklevel=4)
    return _NoNative()


def _bind_native():
    global _native
    load_library()
    torch = _bind_torch()  # the extension's symbols are torch's
    if isinstance(_native, _Unbound):
        native = _load_native(torch)
        _bind_addresses(native)
        _native = native
    return _native


_torch = None
_dtype_codes = {}
_raw_stream = _current_device = _capturing = None


def _bind_torch():
    """torch, imported by the first call that takes tensors (the host-only calls do without)."""
    global _torch, _capturing
    if _torch is None:
        import torch
        _capturing = torch.cuda.is_current_stream_capturing
        _dtype_codes.update({torch.float32: DTYPE_F32, torch.float16: DTYPE_F16})
        _torch = torch
    return _torch


def _dtype_code(t):
    code = _dtype_codes.get(t.dtype)
    if code is None:
        _bind_torch()
        code = _dtype_codes.get(t.dtype)
        if code is None:
            raise MsdError("unsupported storage dtype %s" % t.dtype)
    return code


def _stream():
    """The handle of torch's current stream on the current device.  Two private functions of torch's give it without
    a stream object (0.3 us against 1.6 a call); a torch that lacks them is asked through its public ones."""
    global _raw_stream, _current_device
    if _raw_stream is None:
        torch = _bind_torch()
        handle = torch.cuda.current_stream().cuda_stream  # initialises the device where nothing has yet
        _current_device = getattr(torch._C, "_cuda_getDevice", torch.cuda.current_device)
        _raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None) or \
            (lambda device: torch.cuda.current_stream(device).cuda_stream)
        return handle
    return _raw_stream(_current_device())


def _dev(t):
    if not t.is_cuda or not t.is_contiguous():
        raise MsdError("expected a contiguous device tensor")
    return t.data_ptr()


def _affine(t, n, like, what):
    """gamma / beta / bias: float32, n values, on the device of `like`."""
    if t.dtype != (_torch or _bind_torch()).float32 or t.numel() != n or t.get_device() != like.get_device():
        raise MsdError("%s must be float32 with %d values on %s (got %s, %d, %s)"
                       % (what, n, like.device, t.dtype, t.numel(), t.device))
    return _dev(t)


def _same(t, like, numel, what):
    """An output / second operand: dtype and device of `like`, `numel` elements."""
    if t.dtype != like.dtype or t.get_device() != like.get_device() or t.numel() != numel:
        raise MsdError("%s must be %s with %d elements on %s (got %s, %d, %s)"
                       % (what, like.dtype, numel, like.device, t.dtype, t.numel(), t.device))
    return _dev(t)


def _out_like(x, out, what="out"):
    """(output, its pointer): a new tensor like x, which _dev has checked, or the caller's."""
    if out is None:
        out = (_torch or _bind_torch()).empty_like(x)
        return out, out.data_ptr()
    return out, _same(out, x, x.numel(), what)


def init():
    check(load_library().msd_init(_stream()))


def status():
    return load_library().msd_status(_stream())


def gn_fallbacks(reset=False):
    """How often a GroupNorm workgroup computed a sibling's statistics itself (diagnostic)."""
    n = ctypes.c_uint(0)
    check(load_library().msd_gn_fallbacks(_stream(), ctypes.byref(n), int(reset)))
    return n.value


def _planes(x):
    """(batch, channels, positions per channel) of [batch, C, ...]."""
    shape = x.shape
    batch, channels = shape[0], shape[1]
    return batch, channels, x.numel() // (batch * channels) if batch * channels else 0


def groupnorm(x, gamma, beta, groups, eps=1e-5, fuse_silu=False, out=None, noalloc=False):
    """x: [batch, C, ...] device tensor; gamma/beta float32 [C]; out may be x (in place).
    noalloc: go through msd_groupnorm_noalloc (fixed scratch, batch * groups <= 1024)."""
    done = _native.groupnorm(x, gamma, beta, groups, eps, fuse_silu, out, noalloc)
    if done is not None:
        return done
    lib = _lib or load_library()
    batch, channels, hw = _planes(x)
    xp = _dev(x)
    out, yp = _out_like(x, out)
    check((lib.msd_groupnorm_noalloc if noalloc else lib.msd_groupnorm)(
        xp, yp, _affine(gamma, channels, x, "gamma"), _affine(beta, channels, x, "beta"), batch, channels, hw, groups,
        eps, int(fuse_silu), _dtype_code(x), _stream()))
    return out


def groupnorm_plan(batch, channels, hw, groups=32, dtype_code=DTYPE_F16, noalloc=False, in_place=False):
    """(split, threads, vectors per lane, writers) of the launch msd_groupnorm makes for this
    shape; (0, 0, 0, 1) = the general kernel; writers > 1 = that many workgroups share each whole
    (sample, group) and store a part of it each (never for a call in place).  Host arithmetic,
    no GPU needed."""
    out = [ctypes.c_int(0) for _ in range(4)]
    check(load_library().msd_groupnorm_plan(batch, channels, hw, groups, dtype_code, int(noalloc), int(in_place),
                                            *[ctypes.byref(o) for o in out]))
    return tuple(o.value for o in out)


def groupnorm_tokens(x, gamma, beta, groups, eps=1e-6):
    """x: [batch, C, ...] -> [batch, H*W, C] = GroupNorm(x) with channels last (no SiLU)."""
    done = _native.groupnorm_tokens(x, gamma, beta, groups, eps)
    if done is not None:
        return done
    lib = _lib or load_library()
    batch, channels, hw = _planes(x)
    xp = _dev(x)
    out = x.new_empty((batch, hw, channels))
    gp, bp = _affine(gamma, channels, x, "gamma"), _affine(beta, channels, x, "beta")
    if not _capturing():
        check(lib.msd_groupnorm_tokens(xp, out.data_ptr(), gp, bp, batch, channels, hw, groups, eps, _dtype_code(x),
                                       _stream()))
        return out
    size = TOKENS_WORKSPACE_BYTES * batch * groups
    workspace = x.new_empty(size, dtype=_torch.uint8)  # (the graph keeps it in its pool, apart from other graphs')
    check(lib.msd_groupnorm_tokens_workspace(xp, out.data_ptr(), gp, bp, batch, channels, hw, groups, eps, _dtype_code(x),
                                             workspace.data_ptr(), size, _stream()))
    return out


def permute_0_2_1(x):
    """[i, j, k] -> [i, k, j] (new tensor)."""
    done = _native.permute_0_2_1(x)
    if done is not None:
        return done
    lib = _lib or load_library()
    i, j, k = x.shape
    xp = _dev(x)
    out = x.new_empty((i, k, j))
    check(lib.msd_permute_0_2_1(xp, out.data_ptr(), i, j, k, _dtype_code(x), _stream()))
    return out


def chunk_add_groupnorm(x, chunk, gamma, beta, groups, eps=1e-5, fuse_silu=False, out=None):
    """GroupNorm(x + chunk[:, :, None]) (+ SiLU); chunk: [batch, C] in x's dtype."""
    done = _native.chunk_add_groupnorm(x, chunk, gamma, beta, groups, eps, fuse_silu, out)
    if done is not None:
        return done
    lib = _lib or load_library()
    batch, channels, hw = _planes(x)
    xp = _dev(x)
    cp = _same(chunk, x, batch * channels, "chunk")
    out, yp = _out_like(x, out)
    check(lib.msd_chunk_add_groupnorm(xp, cp, yp, _affine(gamma, channels, x, "gamma"), _affine(beta, channels, x, "beta"),
                                      batch, channels, hw, groups, eps, int(fuse_silu), _dtype_code(x), _stream()))
    return out


def add_layernorm(a, b, gamma, beta, eps=1e-5, sum_out=None, out=None):
    """Returns (a + b, LayerNorm(a + b)); sum_out may be a or b."""
    done = _native.add_layernorm(a, b, gamma, beta, eps, sum_out, out)
    if done is not None:
        return done
    lib = _lib or load_library()
    n, dim = a.numel(), a.shape[-1]
    rows = n // dim if dim else 0
    ap, bp = _dev(a), _same(b, a, n, "b")
    sum_out, sp = _out_like(a, sum_out, "sum_out")
    out, yp = _out_like(a, out)
    check(lib.msd_add_layernorm(ap, bp, sp, yp, _affine(gamma, dim, a, "gamma"), _affine(beta, dim, a, "beta"), rows, dim,
                                eps, _dtype_code(a), _stream()))
    return sum_out, out


def elemwise_add(a, b, out=None):
    done = _native.elemwise_add(a, b, out)
    if done is not None:
        return done
    lib = _lib or load_library()
    n = a.numel()
    ap, bp = _dev(a), _same(b, a, n, "b")
    out, yp = _out_like(a, out)
    check(lib.msd_elemwise_add(ap, bp, yp, n, _dtype_code(a), _stream()))
    return out


def chunkwise_add(a, chunk, chunk_size, out=None):
    done = _native.chunkwise_add(a, chunk, chunk_size, out)
    if done is not None:
        return done
    lib = _lib or load_library()
    n = a.numel()
    if chunk_size <= 0 or n % chunk_size:
        raise MsdError("chunk_size must divide the element count")
    ap, cp = _dev(a), _same(chunk, a, n // chunk_size, "chunk")
    out, yp = _out_like(a, out)
    check(lib.msd_chunkwise_add(ap, cp, yp, n, chunk_size, _dtype_code(a), _stream()))
    return out


def layernorm(x, gamma, beta, eps=1e-5, out=None):
    done = _native.layernorm(x, gamma, beta, eps, out)
    if done is not None:
        return done
    lib = _lib or load_library()
    dim = x.shape[-1]
    rows = x.numel() // dim if dim else 0
    xp = _dev(x)
    out, yp = _out_like(x, out)
    check(lib.msd_layernorm(xp, yp, _affine(gamma, dim, x, "gamma"), _affine(beta, dim, x, "beta"), rows, dim, eps,
                            _dtype_code(x), _stream()))
    return out


def geglu(proj, out=None):
    """proj: [..., 2*inner] (value | gate) -> [..., inner]."""
    done = _native.geglu(proj, out)
    if done is not None:
        return done
    lib = _lib or load_library()
    shape = proj.shape
    inner = shape[-1] // 2
    rows = proj.numel() // (2 * inner) if inner else 0
    pp = _dev(proj)
    if out is None:
        out = proj.new_empty(shape[:-1] + (inner,))
    check(lib.msd_geglu(pp, _same(out, proj, rows * inner, "out"), rows, inner, _dtype_code(proj), _stream()))
    return out


def _act(name, x, out):
    fn = getattr(_lib or load_library(), name)
    xp = _dev(x)
    out, yp = _out_like(x, out)
    check(fn(xp, yp, x.numel(), _dtype_code(x), _stream()))
    return out


def silu(x, out=None):
    done = _native.silu(x, out)
    return done if done is not None else _act("msd_silu", x, out)


def gelu(x, out=None):
    done = _native.gelu(x, out)
    return done if done is not None else _act("msd_gelu", x, out)


def quick_gelu(x, out=None):
    done = _native.quick_gelu(x, out)
    return done if done is not None else _act("msd_quick_gelu", x, out)


def timestep_embedding(timesteps, dim, max_period=10000.0, dtype=None):
    """timesteps: int64 device tensor [batch] -> [batch, dim] as [cos | sin]."""
    torch = _torch or _bind_torch()
    if dtype is None or dtype is torch.float32 or dtype is torch.float16:
        done = _native.timestep_embedding(timesteps, dim, max_period, dtype is torch.float16)
        if done is not None:
            return done
    lib = _lib or load_library()
    n = timesteps.numel()
    out = timesteps.new_empty((n, dim), dtype=dtype or torch.float32)
    check(lib.msd_timestep_embedding(_dev(timesteps), _dev(out), n, dim, max_period, _dtype_code(out), _stream()))
    return out


def ddim_timesteps(steps):
    """Ascending integer DDIM timestep list (host only)."""
    lib = load_library()
    n = lib.msd_ddim_timesteps(steps, None, 0)
    if n < 0:
        raise MsdError("ddim steps must be in [1, 1000]")
    buf = (ctypes.c_int * n)()
    lib.msd_ddim_timesteps(steps, buf, n)
    return list(buf)


def linear_rows(x, weight, bias=None, act_in=ACT_NONE, act_out=ACT_NONE, out=None):
    """x [m <= 8, k], weight [n, k] (x's dtype), bias float32 [n] or None -> [m, n]."""
    done = _native.linear_rows(x, weight, bias, act_in, act_out, out)
    if done is not None:
        return done
    lib = _lib or load_library()
    m, k = x.shape
    n = weight.shape[0]
    if weight.shape[1] != k or weight.dtype != x.dtype:
        raise MsdError("weight must be [n, k] in the dtype of x")
    if weight.get_device() != x.get_device():
        raise MsdError("weight and x must share a device")
    xp, wp = _dev(x), _dev(weight)
    bp = _affine(bias, n, x, "bias") if bias is not None else None
    out = x.new_empty((m, n)) if out is None else out
    check(lib.msd_linear_rows(xp, wp, bp, _same(out, x, m * n, "out"), m, n, k, act_in, act_out, _dtype_code(x), _stream()))
    return out


def linear_rows_grouped(x, weights, biases=None, act_in=ACT_NONE, act_out=ACT_NONE):
    """One launch for several Linear layers on the same x [m <= 8, k]: weights[i] is [n_i, k] in
    x's dtype, biases[i] float32 [n_i] or None -> list of [m, n_i] tensors."""
    done = _native.linear_rows_grouped(x, weights, biases, act_in, act_out)
    if done is not None:
        return done
    lib = _lib or load_library()
    m, k = x.shape
    xp, dtype, device, new = _dev(x), x.dtype, x.get_device(), x.new_empty
    outs, wp, bp, yp, ns = [], [], [], [], []
    for i, w in enumerate(weights):
        shape = w.shape
        if len(shape) != 2 or shape[1] != k or w.dtype != dtype or w.get_device() != device:
            raise MsdError("weights[%d] must be [n, %d] in the dtype and on the device of x" % (i, k))
        n = shape[0]
        b = biases[i] if biases is not None else None
        bp.append(_affine(b, n, x, "biases[%d]" % i) if b is not None else None)
        if not w.is_contiguous():
            raise MsdError("expected contiguous weights")
        out = new((m, n))
        outs.append(out)
        wp.append(w.data_ptr())  # (0 for an empty tensor, as for the others)
        yp.append(out.data_ptr())
        ns.append(n)
    count = len(outs)
    pointers = ctypes.c_void_p * count
    check(lib.msd_linear_rows_grouped(xp, pointers(*wp), pointers(*bp), pointers(*yp), (ctypes.c_size_t * count)(*ns), count,
                                      m, k, act_in, act_out, _dtype_code(x), _stream()))
    return outs


def softmax(x, stable=False, out=None):
    """Softmax over the last axis; out may be x (in place)."""
    done = _native.softmax(x, stable, out)
    if done is not None:
        return done
    lib = _lib or load_library()
    cols = x.shape[-1]
    rows = x.numel() // cols if cols else 0
    xp = _dev(x)
    out, yp = _out_like(x, out)
    check(lib.msd_softmax(xp, yp, rows, cols, int(stable), _dtype_code(x), _stream()))
    return out


def alphas_cumprod():
    """The sampler's 1000 cumulative alpha products as a list of floats (host only)."""
    buf = (ctypes.c_float * 1000)()
    check(load_library().msd_alphas_cumprod(buf))
    return list(buf)


def ddim_schedule(steps):
    """-> (timesteps, alphas, alphas_prev, sqrt_one_minus_alphas) as lists (host only)."""
    lib = load_library()
    n = lib.msd_ddim_schedule(steps, None, None, None, None, 0)
    if n < 0:
        raise MsdError("ddim steps must be in [1, 500] (code %d)" % n)
    ts = (ctypes.c_int * n)()
    a, ap, s1m = (ctypes.c_float * n)(), (ctypes.c_float * n)(), (ctypes.c_float * n)()
    lib.msd_ddim_schedule(steps, ts, a, ap, s1m, n)
    return list(ts), list(a), list(ap), list(s1m)


def ddim_update(x, e_t, a_t, a_prev, sqrt_one_minus_at, out=None):
    """One DDIM step (eta 0) on device tensors; out may be x."""
    done = _native.ddim_update(x, e_t, a_t, a_prev, sqrt_one_minus_at, out)
    if done is not None:
        return done
    lib = _lib or load_library()
    n = x.numel()
    xp, ep = _dev(x), _same(e_t, x, n, "e_t")
    out, yp = _out_like(x, out)
    check(lib.msd_ddim_update(xp, ep, yp, n, a_t, a_prev, sqrt_one_minus_at, _dtype_code(x), _stream()))
    return out


# ---------------------------------------------------------------------------------------
# C++ layer objects (libmsd_nn.so) through their plain-C handles
# ---------------------------------------------------------------------------------------
_nn = None
# int model(void *x, int t, void *e_t, size_t bytes, void *user): the sampler's noise-model callback
MODEL_FN = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p, ctypes.c_size_t,
                            ctypes.c_void_p)


def load_nn_library(path=None):
    """Loads libmsd_nn.so (GroupNorm / LayerNorm / GEGLU objects, NPY loader, step runner)."""
    global _nn
    if _nn is not None and path is None:
        return _nn
    load_library()
    path = path or LIB_NN_PATH
    if not os.path.exists(path):
        raise MsdError("native library %s is missing: run __graft_entry__.build()" % path)
    nn = ctypes.CDLL(path)
    vp, sz, fl, it, cp = ctypes.c_void_p, ctypes.c_size_t, ctypes.c_float, ctypes.c_int, ctypes.c_char_p
    szp = ctypes.POINTER(ctypes.c_size_t)
    flp = ctypes.POINTER(ctypes.c_float)
    lgp = ctypes.POINTER(ctypes.c_long)
    sig = {
        "msdnn_last_error": (cp, []),
        "msdnn_set_media_path": (None, [cp]),
        "msdnn_set_debug_timing": (None, [it]),
        "msdnn_npy_load": (it, [cp, flp, sz, szp, szp]),
        "msdnn_npy_save": (it, [cp, flp, sz]),
        "msdnn_groupnorm_create": (vp, [vp, sz, sz, fl, cp, cp, sz, it]),
        "msdnn_groupnorm_init": (it, [vp]),
        "msdnn_groupnorm_check": (it, [vp, sz, it]),
        "msdnn_groupnorm_forward": (it, [vp, vp, vp, sz, it]),
        "msdnn_groupnorm_forward_chunk": (it, [vp, vp, vp, sz, vp, sz, it]),
        "msdnn_groupnorm_forward_tokens": (it, [vp, vp, vp, sz, it]),
        "msdnn_groupnorm_destroy": (None, [vp]),
        "msdnn_layernorm_create": (vp, [vp, sz, cp, cp, fl]),
        "msdnn_layernorm_init": (it, [vp]),
        "msdnn_layernorm_check": (it, [vp, sz, it]),
        "msdnn_layernorm_forward": (it, [vp, vp, vp, sz, it]),
        "msdnn_layernorm_forward_add": (it, [vp, vp, vp, vp, vp, sz, it]),
        "msdnn_layernorm_destroy": (None, [vp]),
        "msdnn_geglu_create": (vp, [vp, sz, sz]),
        "msdnn_geglu_weight_shape": (it, [vp, szp, szp]),
        "msdnn_geglu_check": (it, [vp, sz, sz, it]),
        "msdnn_geglu_forward": (it, [vp, vp, sz, vp, sz, it]),
        "msdnn_geglu_destroy": (None, [vp]),
        "msdnn_activation": (it, [vp, it, vp, vp, sz, it]),
        "msdnn_timestep_embedding": (it, [vp, lgp, sz, flp]),
        "msdnn_ddim_timesteps": (it, [it, ctypes.POINTER(ctypes.c_int), it]),
        "msdnn_linear_create": (vp, [vp, sz, sz, cp, cp, it]),
        "msdnn_linear_init": (it, [vp]),
        "msdnn_linear_init_from": (it, [vp, flp, sz, flp, sz]),
        "msdnn_linear_forward": (it, [vp, vp, sz, vp, sz, it, it, it]),
        "msdnn_linear_forward_grouped": (it, [ctypes.POINTER(vp), sz, vp, sz, ctypes.POINTER(vp), szp, it, it, it]),
        "msdnn_linear_destroy": (None, [vp]),
        "msdnn_softmax": (it, [vp, vp, vp, sz, it, sz, it]),
        "msdnn_ddim_sample": (it, [vp, vp, sz, it, it, MODEL_FN, vp, vp]),
        "msdnn_ddim_make_schedule": (it, [ctypes.POINTER(ctypes.c_int), it, flp, flp]),
        "msdnn_test_buffer": (it, [vp, vp, sz, it, cp, flp, szp]),
        "msdnn_step_create": (vp, [vp, sz, it, it]),
        "msdnn_step_num_ops": (sz, [vp]),
        "msdnn_step_op_info": (it, [vp, sz, ctypes.POINTER(ctypes.c_int), szp, ctypes.POINTER(ctypes.c_int)]),
        "msdnn_step_download": (it, [vp, sz, it, flp, sz, szp]),
        "msdnn_step_affine": (it, [vp, sz, flp, flp, sz]),
        "msdnn_step_restore": (it, [vp]),
        "msdnn_step_bytes": (sz, [vp]),
        "msdnn_step_launches": (sz, [vp]),
        "msdnn_step_run": (it, [vp, it, it, lgp, sz]),
        "msdnn_step_destroy": (None, [vp]),
    }
    for name, (res, args) in sig.items():
        fn = getattr(nn, name)
        fn.restype = res
        fn.argtypes = args
    _nn = nn
    return nn


def nn_last_error():
    return load_nn_library().msdnn_last_error().decode()
