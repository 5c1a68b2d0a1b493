"""Build the native parts of clode_amd in-tree.

* ``libclode_hip.so``: the HIP runtime and C ABI (include/clode_hip.h).  Host
  C++ compiled with g++ against the HIP runtime and hipRTC; the integration
  kernels are compiled at run time by hipRTC from the device sources that are
  embedded into the library here.
* ``cpp/clode_cpp_wrapper*.so``: the pybind11 module mirroring the
  reference's ``clode.cpp.clode_cpp_wrapper`` over the C ABI.
* ``libclode_mlp.so``: BF16-MFMA surrogate kernels (hipcc, gfx950).
* ``_build/valu_rate``: the FP32/FP64 FMA throughput probe behind
  ``bench.py --calibrate-fma``.

Run ``python clode_amd/build.py`` (or ``__graft_entry__.build()``); it does not
import the clode_amd package, whose import needs the pybind module built here.
"""
from __future__ import annotations

import os
import subprocess
import sys
import sysconfig
from pathlib import Path

PKG = Path(__file__).resolve().parent
CSRC = PKG / "csrc"
DEVICE = CSRC / "device"
RUNTIME = CSRC / "runtime"
REPO = PKG.parent
ROCM = Path(os.environ.get("ROCM_PATH", "/opt/rocm"))

DEVICE_HEADERS = [
    "cm_math.h",
    "clode_builtins.h",
    "clode_divide.h",
    "clode_prelude.h",
    "clode_layout.h",
    "clode_kernel_args.h",
    "clode_rng.h",
    "clode_steppers.h",
    "clode_observers.h",
    "clode_kernels.h",
    "clode_queue.h",
    "clode_system_end.h",
]

HIP_DEVICE_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    # packed FP32 (v_pk_*_f32) is disabled for every device code object
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def _run(cmd: list[str], cwd: Path | None = None) -> None:
    print("+", " ".join(str(c) for c in cmd), flush=True)
    subprocess.run([str(c) for c in cmd], check=True, cwd=cwd)


def embed_device_sources() -> Path:
    """Write runtime/device_sources.inc: the device headers as raw strings."""
    out = RUNTIME / "device_sources.inc"
    lines = ["// generated by clode_amd/build.py from clode_amd/csrc/device/*.h",
             "struct DeviceSource { const char *name; const char *text; };",
             "static const DeviceSource kDeviceSources[] = {"]
    for name in DEVICE_HEADERS:
        path = DEVICE / name
        if not path.exists():
            continue
        text = path.read_text()
        if ')CLODE_SRC"' in text:
            raise RuntimeError(f"{name} contains the raw-string delimiter")
        # split into <= 60 KB chunks (compiler string-literal limits)
        chunks = [text[i:i + 60000] for i in range(0, len(text), 60000)] or [""]
        body = " ".join(f'R"CLODE_SRC({c})CLODE_SRC"' for c in chunks)
        lines.append(f'    {{"{name}", {body}}},')
    lines.append("};")
    content = "\n".join(lines) + "\n"
    if not out.exists() or out.read_text() != content:
        out.write_text(content)
    return out


def build_library() -> Path:
    embed_device_sources()
    out = PKG / "libclode_hip.so"
    srcs = [RUNTIME / "runtime.cpp", RUNTIME / "simulator.cpp", RUNTIME / "batch.cpp", RUNTIME / "capi.cpp"]
    cmd = ["g++", "-O2", "-g", "-fPIC", "-shared", "-std=c++17", "-Wall", "-Wno-unused-function",
           "-Wno-unused-result", "-Wno-stringop-truncation",
           "-D__HIP_PLATFORM_AMD__", f"-I{ROCM / 'include'}", f"-I{REPO / 'include'}",
           *srcs, "-o", out, f"-L{ROCM / 'lib'}", "-lamdhip64", "-lhiprtc",
           f"-Wl,-rpath,{ROCM / 'lib'}"]
    _run(cmd)
    return out


def build_pybind() -> Path:
    import pybind11

    ext = sysconfig.get_config_var("EXT_SUFFIX") or ".so"
    out = PKG / "cpp" / f"clode_cpp_wrapper{ext}"
    src = CSRC / "pybind" / "clode_cpp_wrapper.cpp"
    if not src.exists():
        return out
    py_inc = sysconfig.get_paths()["include"]
    # hidden visibility, as pybind11 recommends for extension modules; the
    # module's init function is exported explicitly
    cmd = ["g++", "-O2", "-fPIC", "-shared", "-std=c++17", "-fvisibility=hidden", f"-I{pybind11.get_include()}",
           f"-I{py_inc}",
           f"-I{REPO / 'include'}", src, "-o", out, f"-L{PKG}", "-lclode_hip", "-Wl,-rpath,$ORIGIN/.."]
    _run(cmd)
    return out


def build_mlp() -> Path | None:
    src = CSRC / "mlp" / "clode_mlp.hip"
    out = PKG / "libclode_mlp.so"
    if not src.exists():
        return None
    cmd = [str(ROCM / "bin" / "hipcc"), *HIP_DEVICE_FLAGS, "-fPIC", "-shared", f"-I{REPO / 'include'}",
           src, "-o", out]
    _run(cmd)
    return out


CALIB_FMA = PKG / "_build" / "valu_rate"


def build_calib() -> Path:
    """The vector-ALU FMA throughput probe run by `bench.py --calibrate-fma`."""
    CALIB_FMA.parent.mkdir(parents=True, exist_ok=True)
    cmd = [str(ROCM / "bin" / "hipcc"), *HIP_DEVICE_FLAGS, CSRC / "calib" / "valu_rate.hip", "-o", CALIB_FMA]
    _run(cmd)
    return CALIB_FMA


def build_all() -> None:
    build_library()
    build_pybind()
    build_mlp()
    build_calib()


if __name__ == "__main__":
    build_all()
    sys.exit(0)
