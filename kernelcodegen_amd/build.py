"""In-tree build of libkcg_hip.so (code generator + hipRTC/hipModule runtime).

    python -m kernelcodegen_amd.build            # build if sources changed
    python -m kernelcodegen_amd.build --force

The kernel templates under csrc/backend/kernels/*.hip are embedded into the
library as raw strings (generated header _templates_gen.inc).  They are device
code for gfx950 only; `check_templates()` cross-compiles every family offline
with hipcc --offload-arch=gfx950 so that a template that no longer compiles
fails the build without needing a GPU.
"""
import glob
import hashlib
import os
import subprocess
import sys
import sysconfig

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
CSRC = os.path.join(PKG, "csrc")
KDIR = os.path.join(CSRC, "backend", "kernels")
LIB = os.path.join(PKG, "libkcg_hip.so")
LAUNCH = os.path.join(PKG, "_launch" + (sysconfig.get_config_var("EXT_SUFFIX") or ".so"))      # another Python does not find it
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
HIPCC = os.path.join(ROCM, "bin", "hipcc")
CXX = os.environ.get("CXX", "g++")

DEVICE_FLAGS = ["--offload-arch=gfx950", "-O3", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]


def sources():
    out = []
    for sub in ("runtime", "capi", "backend", "ir", "frontend", "optimizer", "driver"):
        out += sorted(glob.glob(os.path.join(CSRC, sub, "*.cc")))
    return out


def gen_templates():
    """kernels/*.hip -> kernels/_templates_gen.inc (one raw string each)."""
    parts = ["// generated by kernelcodegen_amd/build.py from kernels/*.hip -- do not edit\n"]
    for path in sorted(glob.glob(os.path.join(KDIR, "*.hip"))):
        name = os.path.splitext(os.path.basename(path))[0]
        text = open(path).read()
        assert ')KCGTPL"' not in text
        parts.append('static const char kTpl_%s[] = R"KCGTPL(%s)KCGTPL";\n' % (name, text))
    new = "".join(parts)
    dst = os.path.join(KDIR, "_templates_gen.inc")
    if not os.path.exists(dst) or open(dst).read() != new:
        with open(dst, "w") as f:
            f.write(new)
    return dst


def _stamp():
    h = hashlib.sha256()
    files = sources() + sorted(glob.glob(os.path.join(KDIR, "*.hip"))) + [os.path.join(CSRC, "runtime", "kcg_scratch.hip")]
    files += sorted(glob.glob(os.path.join(ROOT, "include", "**", "*.h"), recursive=True))
    files += sorted(glob.glob(os.path.join(CSRC, "**", "*.h"), recursive=True))
    for p in files:
        h.update(p.encode())
        h.update(open(p, "rb").read())
    return h.hexdigest()


def build_launch(force=False, verbose=False):
    """The bound launches of the Python operators (launch.cc), an extension module on torch's own libraries; None where there is no
    torch to build it on or the compiler refuses it, whose messages are shown: ctypes launches take its place."""
    stamp_file = LAUNCH + ".stamp"
    try:
        import torch
        src = os.path.join(os.path.dirname(CSRC), "launch.cc")
        base = os.path.dirname(torch.__file__)
        inc = os.path.join(base, "include")
        cmd = [CXX, "-std=c++17", "-O2", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
               "-D_GLIBCXX_USE_CXX11_ABI=%d" % torch._C._GLIBCXX_USE_CXX11_ABI, '-DKCG_TORCH_VERSION="%s"' % torch.__version__,
               "-I", inc, "-I", os.path.join(inc, "torch", "csrc", "api", "include"),
               "-I", os.path.join(ROCM, "include"), "-I", sysconfig.get_paths()["include"], src, "-o", LAUNCH, "-L", os.path.join(base, "lib"),
               "-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10", "-lc10_hip"]
        stamp = hashlib.sha256((open(src).read() + " ".join(cmd)).encode()).hexdigest()
        if not force and os.path.exists(LAUNCH) and os.path.exists(stamp_file) and open(stamp_file).read() == stamp:
            return LAUNCH
        if verbose:
            print(" ".join(cmd))
        done = subprocess.run(cmd, stderr=subprocess.PIPE, text=True, errors="replace")
        why = "%s\nstatus %d" % (done.stderr, done.returncode) if done.returncode else ""
    except (ImportError, OSError) as e:
        why = str(e)
    if why:
        for stale in (LAUNCH, stamp_file):
            if os.path.exists(stale):
                os.remove(stale)
        print("%s\nthe native launches were not built: launches go through ctypes" % why, file=sys.stderr)
        return None
    with open(stamp_file, "w") as f:
        f.write(stamp)
    return LAUNCH


def build(force=False, verbose=False):
    """libkcg_hip.so, then the native launches where they can be built; returns the library."""
    library = build_library(force, verbose)
    build_launch(force, verbose)
    return library


def build_library(force=False, verbose=False):
    gen_templates()
    stamp_file = LIB + ".stamp"
    stamp = _stamp()
    if not force and os.path.exists(LIB) and os.path.exists(stamp_file) and open(stamp_file).read() == stamp:
        return LIB
    # The one file with device code (the scratch array of kcg_hip_launch_scratch and its clearing kernel) is
    # compiled by hipcc for gfx950; everything else is host code (the kernels proper are emitted at run time), so
    # the system C++ compiler builds it; the library links the HIP runtime and opens hipRTC itself (dlmopen).
    scratch_obj = os.path.join(CSRC, "runtime", "kcg_scratch.o")
    cmd = [HIPCC] + DEVICE_FLAGS + ["-std=c++17", "-fPIC", "-c", "-I", os.path.join(ROOT, "include"), "-I", CSRC,
                                    os.path.join(CSRC, "runtime", "kcg_scratch.hip"), "-o", scratch_obj]
    if verbose:
        print(" ".join(cmd))
    subprocess.check_call(cmd, stderr=None if verbose else subprocess.DEVNULL)
    # One object per translation unit, compiled side by side and kept under csrc/_obj: a change to one source file
    # recompiles that file, a change to any header all of them (`force` too).
    from concurrent.futures import ThreadPoolExecutor
    objdir = os.path.join(CSRC, "_obj")
    os.makedirs(objdir, exist_ok=True)
    headers = sorted(glob.glob(os.path.join(ROOT, "include", "**", "*.h"), recursive=True))
    headers += sorted(glob.glob(os.path.join(CSRC, "**", "*.h"), recursive=True))
    headers += [os.path.join(KDIR, "_templates_gen.inc")]
    hh = hashlib.sha256()
    for p in headers:
        hh.update(open(p, "rb").read())
    flags = [CXX, "-std=c++17", "-O2", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-Wall", "-Wno-unused-function",
             "-Wno-init-list-lifetime", "-I", os.path.join(ROOT, "include"), "-I", CSRC, "-I", os.path.join(ROCM, "include")]

    def compile_one(src):
        tag = os.path.relpath(src, CSRC).replace(os.sep, "__")
        obj = os.path.join(objdir, tag + ".o")
        key = hashlib.sha256(hh.digest() + open(src, "rb").read() + " ".join(flags).encode()).hexdigest()
        keyfile = obj + ".key"
        if force or not os.path.exists(obj) or not os.path.exists(keyfile) or open(keyfile).read() != key:
            cmd = flags + ["-c", src, "-o", obj]
            if verbose:
                print(" ".join(cmd))
            subprocess.check_call(cmd)
            with open(keyfile, "w") as f:
                f.write(key)
        return obj

    with ThreadPoolExecutor(max_workers=min(8, os.cpu_count() or 1)) as pool:
        objs = list(pool.map(compile_one, sources()))
    cmd = [CXX, "-shared", "-o", LIB] + objs + [scratch_obj, "-L", os.path.join(ROCM, "lib"), "-lamdhip64", "-ldl",
                                                "-Wl,-rpath," + os.path.join(ROCM, "lib")]
    if verbose:
        print(" ".join(cmd))
    subprocess.check_call(cmd)
    with open(stamp_file, "w") as f:
        f.write(stamp)
    return LIB


def compile_source_offline(src, out_path):
    """hipcc cross-compile of emitted source text to a gfx950 code object."""
    tmp = out_path + ".hip"
    with open(tmp, "w") as f:
        f.write(src)
    subprocess.check_call([HIPCC] + DEVICE_FLAGS + ["--genco", "-o", out_path, tmp],
                          stderr=subprocess.DEVNULL)
    os.remove(tmp)
    return out_path


def prebuild_kernels(verbose=False, force=False):
    """Emit and compile (hipRTC, gfx950, no GPU needed) every benchmark kernel
    into the on-disk code-object cache; `force` compiles also what the cache holds."""
    from . import runtime as R
    from .configs import WORKLOADS, workload_source
    out = []
    for name in WORKLOADS:
        source = workload_source(name)[0]
        code = R.compile_to_code(source, refresh=force)
        out.append((name, len(code)))
        if verbose:
            print("prebuilt %-32s %7d bytes" % (name, len(code)))
    return out


if __name__ == "__main__":
    build(force="--force" in sys.argv, verbose=True)
    print(LIB)
    prebuild_kernels(verbose=True)
