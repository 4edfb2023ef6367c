"""Compiles lact_amd/csrc into lact_amd/lib: liblact_hip.so for gfx950 with hipcc (cross-compiles without a GPU) and
_lact_host.so, the host module between PyTorch and it, with the host compiler.  Usage: python -m lact_amd.build"""
import os
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "csrc", "lact_api.hip")
LIB_DIR = os.path.join(HERE, "lib")
LIB = os.path.join(LIB_DIR, "liblact_hip.so")
HOST_SRC = os.path.join(HERE, "csrc", "torch_host.cpp")
HOST_LIB = os.path.join(LIB_DIR, "_lact_host.so")

FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared",
    # packed-fp32 VALU forms are kept out of the generated code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # A multiply and an add fuse only where one source expression writes them together.  HIP's default ("fast") also
    # fuses across statements and inlined calls, i.e. through __fmul_rn / __fadd_rn, which are plain operators in the
    # HIP headers: whether a product that the reference rounds as a tensor of its own (a * X before + B @ X,
    # ttt_operation.py:62; M * m before dw +, :174-176) got its own rounding then depended on how the surrounding
    # kernel was inlined -- the fused and the unfused Newton-Schulz backward differed in exactly that.
    "-ffp-contract=on",
    # the copy engine sets m0 in its own asm statements and names it as clobbered; no compiler-generated code in these
    # kernels uses m0 (no LDS-DMA builtins, no register-indexed moves, no messages)
    "-Wno-inline-asm",
]


def _host_commands():
    """Compile and link command of the host module (the link needs liblact_hip.so)."""
    import torch
    from torch.utils.cpp_extension import include_paths
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    obj = os.path.join(LIB_DIR, "torch_host.o")
    incs = [f"-I{p}" for p in include_paths() + [os.path.join(rocm, "include"), sysconfig.get_paths()["include"]]]
    cxx = os.environ.get("CXX", "g++")
    compile_ = [cxx, "-O2", "-std=c++17", "-fPIC", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", "-DTORCH_EXTENSION_NAME=_lact_host",
                f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}"] + incs + ["-c", HOST_SRC, "-o", obj]
    torch_lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    link = [cxx, "-shared", obj, "-o", HOST_LIB, f"-L{LIB_DIR}", "-l:liblact_hip.so", f"-L{torch_lib}", "-lc10", "-lc10_hip", "-ltorch",
            "-ltorch_cpu", "-ltorch_hip", "-ltorch_python", "-Wl,-rpath,$ORIGIN"]
    return compile_, link


def build(verbose: bool = True) -> str:
    os.makedirs(LIB_DIR, exist_ok=True)
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    compile_, link = _host_commands()
    cmds = [[hipcc] + FLAGS + [SRC, "-o", LIB], compile_]
    if verbose:
        for cmd in cmds:
            print(" ".join(cmd), flush=True)
    # the device library and the host module compile side by side
    procs = [subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True) for cmd in cmds]
    outs = [p.communicate()[0] for p in procs]
    if all(p.returncode == 0 for p in procs):
        res = subprocess.run(link, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
        procs.append(res)
        outs.append(res.stdout)
    for cmd, p, text in zip(cmds + [link], procs, outs):
        text = "\n".join(l for l in text.splitlines() if "packed-fp32-ops" not in l)
        if p.returncode != 0:
            raise RuntimeError(f"{cmd[0]} failed:\n" + text)
        if verbose and text.strip():
            print(text)
    os.remove(os.path.join(LIB_DIR, "torch_host.o"))
    return LIB


if __name__ == "__main__":
    build()
    sys.exit(0)
