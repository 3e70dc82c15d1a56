"""Compiles the HIP sources of this package into pam_amd/lib/libpam_hip.so for gfx950, and the ops' host path into the
Python module pam_amd/lib/_pam_host.so on top of it.

hipcc cross-compiles without a GPU, so this runs anywhere the ROCm toolchain is installed.
Packed-fp32 instruction selection is switched off and floating-point contraction is off:
the kernels' results are defined operation by operation.
"""
import concurrent.futures
import hashlib
import pathlib
import re
import shutil
import subprocess
import sys
import tempfile

HERE = pathlib.Path(__file__).resolve().parent
CSRC = HERE / "csrc"
SOURCES = [CSRC / "pam_rowops_plain.hip", CSRC / "pam_rowops_offset.hip"] + sorted(CSRC.glob("pam_gemm_inst_*.hip")) + [
    CSRC / "pam_gemm.hip", CSRC / "pam_elementwise.hip", CSRC / "pam_rowops.hip", CSRC / "pam_colsum.hip", CSRC / "pam_probe.hip"]   # slowest first
JOBS = 8
STAMP_SOURCE = CSRC / "pam_stamp.cpp"
HOST_SOURCE = CSRC / "pam_host.cpp"
LIB = HERE / "lib" / "libpam_hip.so"
HOST = HERE / "lib" / "_pam_host.so"

FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]
_NOISE = "is not a recognized feature for this target"      # the host pass does not know the device feature
_TAG = b"pam_hip_source_hash="
_HOST_TAG = b"pam_host_build="


def _host_flags():
    import sysconfig

    import torch
    root = pathlib.Path(torch.__file__).resolve().parent
    flags = ["-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__", "-DTORCH_EXTENSION_NAME=_pam_host",
             f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-I" + sysconfig.get_paths()["include"],
             f"-I{root}/include", f"-I{root}/include/torch/csrc/api/include", "-I/opt/rocm/include"]
    link = [f"-L{root}/lib", "-lc10", "-lc10_hip", "-ltorch", "-ltorch_cpu", "-ltorch_hip", "-ltorch_python", f"-L{LIB.parent}",
            "-l:libpam_hip.so", "-Wl,-rpath,$ORIGIN"]
    return flags, link


def host_hash():
    """Hash of what the host module depends on beside the library's sources: its flags and link line, the torch whose
    headers and libraries it is built on, and the Python it is a module of.  It is compiled into the module."""
    import sysconfig

    import torch
    flags, link = _host_flags()
    parts = [part for part in flags + link if "/" not in part]           # (not where this tree or torch lie)
    parts += [torch.__version__, str(torch.version.git_version), str(sysconfig.get_config_var("SOABI"))]
    return hashlib.sha256("\0".join(parts).encode()).hexdigest()[:16]


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    err = "\n".join(l for l in res.stderr.splitlines() if _NOISE not in l)
    if res.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed:\n" + err)
    if verbose and err.strip():
        print(err, file=sys.stderr)


def _with_includes(src, seen=None):
    """src and the project headers it includes ("..." includes, followed recursively), in a fixed order."""
    seen = [] if seen is None else seen
    src = src.resolve()
    if src in seen or not src.is_file():
        return seen
    seen.append(src)
    for name in re.findall(r'^\s*#\s*include\s+"([^"]+)"', src.read_text(), flags=re.M):
        _with_includes(src.parent / name, seen)
    return seen


def source_files():
    """What the library is built from: the HIP / C++ sources and headers under csrc/ and the public headers.
    Anything else lying in those folders (editor backups, objects, folders) is not part of it."""
    files = [f for pat in ("*.hip", "*.cpp", "*.h") for f in CSRC.glob(pat)] + list((HERE.parent / "include").glob("*.h"))
    return sorted(f for f in files if f.is_file())


def source_hash():
    """Hash of everything the library is built from (source_files() and the compiler flags).  It is compiled
    into the library (pam_hip_source_hash), so a library can be told from one built from other sources."""
    h = hashlib.sha256(" ".join(FLAGS).encode())
    for f in source_files():
        h.update(f.name.encode() + b"\0" + f.read_bytes())
    return h.hexdigest()[:16]


def _stamped(path, tag):
    m = re.search(re.escape(tag) + rb"([0-9a-f]{16})\0", path.read_bytes()) if path.exists() else None
    return m.group(1).decode() if m else None


def built_hash():
    """The hash the built library and host module carry, or None if one is missing, without a stamp or not built with
    the other, or if the module was built on another torch or Python or with other flags.  Read from the files' bytes:
    loading a possibly stale library into this process, which may go on to load its replacement, would register two
    copies of the code objects."""
    found = {_stamped(lib, _TAG) for lib in (LIB, HOST)}
    return found.pop() if len(found) == 1 and _stamped(HOST, _HOST_TAG) == host_hash() else None


def ensure_built(verbose=False):
    """What tests, the smoke check and the benchmark call: the library that is built is used as it is when it was
    built from this tree's sources; a missing or stale one is rebuilt where hipcc is at hand, and is an error where
    it is not.  Returns (path, hash)."""
    want = source_hash()
    have = built_hash()
    if have != want:
        if shutil.which("hipcc") is None:
            raise RuntimeError(f"{LIB} is missing or was built from other sources (want {want}, have {have}) and there is no hipcc to rebuild it")
        build(verbose)
        if built_hash() != want:
            raise RuntimeError("the library just built does not carry the hash of the sources")
    return LIB, want


def build(verbose=False, object_dir=None):
    """Compiles the sources side by side (the matrix kernel's many instances dominate), then links: the library, which
    needs hipcc alone, and then the host module on top of it, which needs g++ and torch's and Python's headers too.
    object_dir: keep the objects there and recompile only the sources that changed since (for development;
    the default compiles everything)."""
    LIB.parent.mkdir(exist_ok=True)
    stamp = f'-DPAM_HIP_SOURCE_HASH="{source_hash()}"'
    with tempfile.TemporaryDirectory() as tmp:
        out = pathlib.Path(object_dir) if object_dir else pathlib.Path(tmp)
        out.mkdir(parents=True, exist_ok=True)

        def compile_one(src, compiler, flags):
            obj, keyfile = out / (src.stem + ".o"), out / (src.stem + ".key")
            key = hashlib.sha256(" ".join(flags).encode() + b"".join(f.read_bytes() for f in _with_includes(src))).hexdigest()
            if not (object_dir and obj.exists() and keyfile.exists() and keyfile.read_text() == key):
                keyfile.unlink(missing_ok=True)
                _run([compiler, *flags, "-c", str(src), "-o", str(obj)], verbose)
                if object_dir:
                    keyfile.write_text(key)
            return str(obj)

        def compile_host():
            flags, link = _host_flags()
            return compile_one(HOST_SOURCE, "g++", flags + [f'-DPAM_HOST_BUILD="{host_hash()}"']), link

        with concurrent.futures.ThreadPoolExecutor(JOBS) as pool:
            jobs = [pool.submit(compile_one, src, "hipcc", FLAGS + ([stamp] if src == STAMP_SOURCE else [])) for src in SOURCES + [STAMP_SOURCE]]
            host_job = pool.submit(compile_host)
            objects = [job.result() for job in jobs]
            _run(["hipcc", "--offload-arch=gfx950", "-shared", "-fPIC", *objects, "-o", str(LIB)], verbose)
            HOST.unlink(missing_ok=True)             # (never beside a library it was not built with)
            host_object, host_link = host_job.result()
        _run(["g++", "-shared", host_object, objects[-1], "-o", str(HOST), *host_link], verbose)
    return LIB


if __name__ == "__main__":
    print(build(verbose=True, object_dir=sys.argv[1] if len(sys.argv) > 1 else None))
