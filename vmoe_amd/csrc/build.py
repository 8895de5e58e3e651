"""Builds libvmoe_hip.so for gfx950 with hipcc (run: python -m vmoe_amd.csrc.build)."""
from __future__ import annotations

import concurrent.futures
import os
import shutil
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
OUT_DIR = os.path.join(os.path.dirname(HERE), "_lib")
LIB = os.path.join(OUT_DIR, "libvmoe_hip.so")
HOST = os.path.join(OUT_DIR, "_vmoe_host.so")      # the host side on torch tensors (host.cpp)
SOURCES = ["capi.hip", "gate_topk.hip", "route_assign.hip", "dispatch_combine.hip",
           "expert_mlp.hip", "soft_moe.hip", "vit_ops.hip"]
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
         "-Wno-unknown-warning-option", "-Wno-unused-command-line-argument",
         "-I", os.path.join(ROOT, "include"), "-I", HERE]


def _hipcc() -> str:
  for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", "hipcc"):
    if cand and (os.path.sep not in cand or os.path.exists(cand)):
      return cand
  raise RuntimeError("hipcc not found")


def _compile(src: str) -> str:
  obj = os.path.join(OUT_DIR, "obj", src.replace(".hip", ".o"))
  cmd = [_hipcc(), *FLAGS, "-c", os.path.join(HERE, src), "-o", obj]
  r = subprocess.run(cmd, capture_output=True, text=True)
  if r.returncode != 0:
    raise RuntimeError(f"hipcc failed on {src}:\n{r.stderr}")
  noise = "is not a recognized feature"
  err = "\n".join(l for l in r.stderr.splitlines() if noise not in l and l.strip())
  if err:
    sys.stderr.write(err + "\n")
  return obj


def _run(cmd, what: str) -> None:
  r = subprocess.run(cmd, capture_output=True, text=True)
  if r.returncode != 0:
    raise RuntimeError(f"{what} failed:\n{r.stderr}")


def _compile_host() -> str:
  """host.cpp: plain C++ against torch's headers (no device code in it)."""
  import torch
  from torch.utils import cpp_extension
  obj = os.path.join(OUT_DIR, "obj", "host.o")
  rocm = os.path.join(os.path.dirname(os.path.dirname(os.path.realpath(shutil.which(_hipcc()) or _hipcc()))), "include")
  includes = [os.path.join(ROOT, "include"), *cpp_extension.include_paths(), rocm,
              sysconfig.get_paths()["include"]]
  _run(["g++", "-O2", "-std=c++17", "-fPIC", "-DTORCH_EXTENSION_NAME=_vmoe_host",
        "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM",       # (c10's stream header declares HIP's types)
        f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
        *[a for i in includes for a in ("-isystem" if "torch" in i else "-I", i)],
        "-c", os.path.join(HERE, "host.cpp"), "-o", obj], "g++ on host.cpp")
  return obj


def _link_host(obj: str) -> None:
  from torch.utils import cpp_extension
  libs = [a for d in cpp_extension.library_paths() for a in ("-L", d)]
  _run(["g++", "-shared", obj, "-o", HOST, *libs, "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch", "-ltorch_python",
        "-L", OUT_DIR, "-l:libvmoe_hip.so", "-Wl,-rpath,$ORIGIN"], "linking the host module")


def build(verbose: bool = True) -> str:
  """Compiles every source and links the shared libraries. Always recompiles."""
  os.makedirs(os.path.join(OUT_DIR, "obj"), exist_ok=True)
  with concurrent.futures.ThreadPoolExecutor(max_workers=min(8, os.cpu_count() or 1)) as ex:
    host = ex.submit(_compile_host)
    objs = list(ex.map(_compile, SOURCES))
    host = host.result()
  cmd = [_hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB, *objs]
  r = subprocess.run(cmd, capture_output=True, text=True)
  if r.returncode != 0:
    raise RuntimeError(f"link failed:\n{r.stderr}")
  _link_host(host)
  if verbose:
    print(f"built {LIB}")
  return LIB


if __name__ == "__main__":
  build()
