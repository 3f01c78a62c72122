"""Build libponni_hip.so (gfx950) in-tree with hipcc.

Every HIP source is compiled for gfx950 only, with packed-fp32 VALU ops
disabled (the compiler otherwise fuses scalar fp32 pairs into v_pk_* forms),
and linked into ponni_amd/libponni_hip.so next to this file.
"""
from __future__ import annotations

import concurrent.futures
import os
import subprocess
import sys
from pathlib import Path

HERE = Path(__file__).resolve().parent
CSRC = HERE / "csrc"
OBJ = HERE / "_build"
LIB = HERE / "libponni_hip.so"
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

SOURCES = [
    "plan.cpp",
    "file_abi.cpp",
    "kernels_generic.hip",
    "kernels_layered.hip",
    "kernels_narrow.hip",
    "kernels_mfma_dispatch.cpp",
    "kernels_mfma_f32_mt2.hip",
    "kernels_mfma_f32_mt4.hip",
    "kernels_mfma_f32_mt8.hip",
    "kernels_fill.hip",
    "fused.cpp",
    "host_exec.cpp",
    "static_scratch.hip",
    "kernels_gather.hip",
    "kernels_peaks.hip",
]

# Headers embedded in the library for the run-time (hipRTC) compiler.
JIT_HEADERS = ["program.h", "pointwise.h", "fused_f32.h", "fused_f16.h", "fused_split.h", "narrow_jit.h"]

COMMON = [
    "-O3",
    "-std=c++20",
    "-fPIC",
    "--offload-arch=gfx950",
    # multiply-adds fuse within one expression only: each layer's state is
    # rounded before the next layer reads it (as the generated kernels)
    "-ffp-contract=on",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall",
    "-Wno-unused-result",
]


def _compile(src: Path, obj: Path) -> None:
    cmd = [HIPCC, *COMMON, "-c", str(src), "-o", str(obj)]
    if src.suffix == ".cpp":
        cmd[1:1] = ["-x", "hip"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src.name}:\n{res.stderr[-6000:]}")


def _write_jit_headers() -> Path:
    out = OBJ / "jit_headers.cpp"
    parts = ["// generated by build.py: headers for the hipRTC-compiled fused kernels",
             "namespace ponni_hip {"]
    names, texts = [], []
    for i, h in enumerate(JIT_HEADERS):
        text = (CSRC / h).read_text()
        assert ")PONNI_SRC" not in text
        parts.append(f'static char const kText{i}[] = R"PONNI_SRC({text})PONNI_SRC";')
        names.append(f'"{h}"')
        texts.append(f"kText{i}")
    parts.append(f"extern char const* const kJitHeaderNames[] = {{{', '.join(names)}}};")
    parts.append(f"extern char const* const kJitHeaderTexts[] = {{{', '.join(texts)}}};")
    parts.append(f"extern int const kJitHeaderCount = {len(JIT_HEADERS)};")
    parts.append("}  // namespace ponni_hip\n")
    text = "\n".join(parts)
    if not out.exists() or out.read_text() != text:
        out.write_text(text)
    return out


def build_library(jobs: int | None = None, verbose: bool = True) -> Path:
    OBJ.mkdir(exist_ok=True)
    jit = _write_jit_headers()
    jobs = jobs or min(8, os.cpu_count() or 4)
    objs = []
    with concurrent.futures.ThreadPoolExecutor(max_workers=jobs) as pool:
        futs = []
        for name in SOURCES:
            src = CSRC / name
            obj = OBJ / (name + ".o")
            objs.append(obj)
            futs.append(pool.submit(_compile, src, obj))
        futs.append(pool.submit(_compile, jit, OBJ / "jit_headers.cpp.o"))
        objs.append(OBJ / "jit_headers.cpp.o")
        for f in futs:
            f.result()
    tmp = LIB.with_suffix(".so.tmp")
    cmd = [HIPCC, "-shared", "-fPIC", "--offload-arch=gfx950", *map(str, objs), "-lhiprtc", "-o", str(tmp)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stderr[-6000:]}")
    os.replace(tmp, LIB)
    if verbose:
        print(f"built {LIB}", file=sys.stderr)
    return LIB


if __name__ == "__main__":
    build_library()
