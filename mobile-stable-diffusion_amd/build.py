"""Build recipe for the native libraries (hipcc cross-compiles gfx950 without a GPU).

    libmsd_hip.so   HIP kernels + the C ABI declared in include/msd_hip.h
    libmsd_nn.so    C++ host layer objects (GroupNorm / LayerNorm / GEGLU / ...) on top of it
    msd_torch_calls.so  the package's calls for plain torch tensors (a CPython extension, host only)
    cli/msd_compare golden-file comparison tool (host only)
    cli/msd_layer_check  runs the layer objects against golden .npy files (needs a GPU)

Run as a script (`python build.py`) or call build_all().
"""
import importlib.util
import os
import subprocess
import sys
import sysconfig

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(PKG_DIR, "csrc")
REPO = os.path.dirname(PKG_DIR)

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"
# -packed-fp32-ops is switched off: plain float code must not be turned into
# v_pk_*_f32 instructions.
# Kernel arguments come in scalar registers, as many as there is room for (the leading ones: pointers and plain
# values, up to the first structure), loaded by the command processor while it prepares the launch.  Otherwise a wavefront's
# first act is to load them, and in a step of 200 launches, each with arguments of its own, that is a miss of every cache in
# front of the launch's first access to its data.  Recorded steps of 512 x 512, us, loaded by the wavefronts and so: fp16
# batch 2 780 -> 753, fp32 batch 1 788 -> 760.  (Launches below 2 us in a row - empty ones, copies, SiLU, DDIM updates of up to
# 0.6 MB - get 0.05 - 0.15 us slower each: the preload is part of what the next one waits for.  Behind a longer launch the same
# ones take as much as before or 0.1 less, and from 2 MB on they get 0.04 faster even where the arguments are in a cache.)
DEVICE_FLAGS = [
    "-O3", "-std=c++17", f"--offload-arch={ARCH}", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-mllvm", "-amdgpu-kernarg-preload-count=16",
    "-Wno-unused-command-line-argument",
]

LIB_HIP = os.path.join(CSRC, "libmsd_hip.so")
LIB_NN = os.path.join(CSRC, "libmsd_nn.so")
TORCH_CALLS = os.path.join(CSRC, "msd_torch_calls.so")
CLI_COMPARE = os.path.join(CSRC, "cli", "msd_compare")
CLI_LAYER_CHECK = os.path.join(CSRC, "cli", "msd_layer_check")


def _run(cmd):
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in proc.stdout.splitlines()
                    if "is not a recognized feature for this target" not in l)
    if proc.returncode != 0:
        raise RuntimeError("build failed: %s\n%s" % (" ".join(cmd), out))
    return out


HIP_SOURCES = ["api.hip", "gn_plan.hip", "groupnorm.hip", "layernorm.hip", "stream_ops.hip", "embed_ops.hip"]


def build_hip():
    """Compiles each translation unit to an object (in parallel) and links libmsd_hip.so."""
    from concurrent.futures import ThreadPoolExecutor
    objs = [os.path.join(CSRC, s.replace(".hip", ".o")) for s in HIP_SOURCES]

    def compile_one(pair):
        src, obj = pair
        return _run([HIPCC] + DEVICE_FLAGS + ["-c", "-o", obj, os.path.join(CSRC, src)])

    with ThreadPoolExecutor(max_workers=6) as pool:
        list(pool.map(compile_one, zip(HIP_SOURCES, objs)))
    _run([HIPCC, "-shared", "-fPIC", f"--offload-arch={ARCH}", "-Wno-unused-command-line-argument",
          "-o", LIB_HIP] + objs)
    return LIB_HIP


def build_nn():
    nn_dir = os.path.join(CSRC, "nn")
    srcs = sorted(os.path.join(nn_dir, f) for f in os.listdir(nn_dir) if f.endswith(".cpp"))
    if not srcs:
        return None
    # host-only C++ against the HIP runtime API: the system compiler, no device code
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared",
           "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include", "-I", os.path.join(REPO, "include"),
           "-I", nn_dir, "-Wall", "-Wno-deprecated-declarations"] + srcs + [
           "-o", LIB_NN, "-L", CSRC, "-lmsd_hip", "-L/opt/rocm/lib", "-lamdhip64",
           "-Wl,-rpath,$ORIGIN", "-Wl,-rpath,/opt/rocm/lib"]
    _run(cmd)
    return LIB_NN


def torch_with_hip_headers():
    """The folder of the installed torch, or None where there is none or it has no HIP headers.  (Does not import it.)"""
    spec = importlib.util.find_spec("torch")
    torch_dir = spec.submodule_search_locations[0] if spec is not None and spec.submodule_search_locations else None
    return torch_dir if torch_dir and os.path.isdir(os.path.join(torch_dir, "include", "ATen", "hip")) else None


def _runs_with(torch_dir):
    """The Python and the torch that torch_calls.cpp is compiled for, as the package asks for them (_running in __init__.py)."""
    spec = importlib.util.spec_from_file_location("torch_version", os.path.join(torch_dir, "version.py"))
    version = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(version)
    return "Python %d.%d, torch %s (%s)" % (sys.version_info[:2] + (version.__version__, version.git_version))


def build_torch_calls():
    """msd_torch_calls.so: host C++ against the headers and libraries of the torch that will import it; None where there is no
    such torch, which nothing else here needs.  NDEBUG, as torch itself is built: without it pybind11's headers give the library
    a thread-local counter that nothing here reads, and glibc takes the slow path of every thread-local access of a process
    (torch's and the runtime's among them) until the thread has touched those of the library loaded last (torch.empty 1.26 us
    against 1.00)."""
    torch_dir = torch_with_hip_headers()
    if torch_dir is None:
        return None
    _run([os.environ.get("CXX", "g++"), "-O2", "-DNDEBUG", "-std=c++17", "-fPIC", "-shared", "-DUSE_ROCM", "-D__HIP_PLATFORM_AMD__",
          '-DMSD_BUILT_FOR="%s"' % _runs_with(torch_dir),
          "-Wall", "-Wno-deprecated-declarations", "-isystem", os.path.join(torch_dir, "include"),
          "-isystem", "/opt/rocm/include", "-isystem", sysconfig.get_paths()["include"],
          os.path.join(CSRC, "torch_calls.cpp"), "-o", TORCH_CALLS, "-L", os.path.join(torch_dir, "lib"), "-ltorch_python",
          "-ltorch_cpu", "-ltorch_hip", "-lc10", "-lc10_hip", "-L/opt/rocm/lib", "-lamdhip64"])
    return TORCH_CALLS


def build_cli():
    """msd_compare: host-only golden-file comparison tool (no HIP, no GPU)."""
    nn_dir = os.path.join(CSRC, "nn")
    _run([os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-Wall", "-I", nn_dir,
          os.path.join(CSRC, "cli", "msd_compare.cpp"), os.path.join(nn_dir, "npy.cpp"), "-o", CLI_COMPARE])
    return CLI_COMPARE


def build_layer_check():
    """msd_layer_check: the layer objects against golden .npy files, from C++ alone."""
    nn_dir = os.path.join(CSRC, "nn")
    _run([os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-Wall", "-Wno-deprecated-declarations",
          "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include", "-I", os.path.join(REPO, "include"), "-I", nn_dir,
          os.path.join(CSRC, "cli", "msd_layer_check.cpp"), "-o", CLI_LAYER_CHECK, "-L", CSRC, "-lmsd_nn",
          "-lmsd_hip", "-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath,$ORIGIN/..", "-Wl,-rpath,/opt/rocm/lib"])
    return CLI_LAYER_CHECK


def build_all(verbose=True):
    built = [build_hip()]
    nn = build_nn()
    if nn:
        built.append(nn)
    built.append(build_cli())
    if nn:
        built.append(build_layer_check())
    torch_calls = build_torch_calls()
    if torch_calls:
        built.append(torch_calls)
    if verbose:
        for b in built:
            print("built", b)
        if not torch_calls:
            print("skipped", TORCH_CALLS, "(no torch with HIP headers here)")
    return built


if __name__ == "__main__":
    build_all()
    sys.exit(0)
