"""Builds what calls the library on PyTorch tensors without the interpreter in between:

    python mops_amd/csrc/build_torch_ops.py

mops_amd/csrc/torch_ops.cpp -> mops_amd/lib/libmops_amd_torch.so, the operators torch.ops.mops.*
(mops_amd/torch.py registers them from Python where it is missing), and mops_amd/csrc/array_ops.cpp
-> mops_amd/lib/_array_ops.so, the functions of the package (mops_amd/ops.py goes through ctypes
where it is missing). Host code only (g++): both call libmops.so, which holds the HIP kernels, and
link against the PyTorch this interpreter imports.
"""
import os
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
LIBRARY_DIR = os.path.join(ROOT, "mops_amd", "lib")
OUTPUTS = {
    "torch_ops.cpp": os.path.join(LIBRARY_DIR, "libmops_amd_torch.so"),
    "array_ops.cpp": os.path.join(LIBRARY_DIR, "_array_ops.so"),
}


def build():
    import torch
    from torch.utils import cpp_extension

    if not os.path.exists(os.path.join(LIBRARY_DIR, "libmops.so")):
        raise RuntimeError("build mops_amd/lib/libmops.so first (make -C mops_amd/csrc)")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    torch_lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    build_dir = os.path.join(HERE, "build")
    os.makedirs(build_dir, exist_ok=True)
    includes = [os.path.join(ROOT, "include"), HERE, os.path.join(rocm, "include")] + cpp_extension.include_paths()
    running = []
    for source, output in OUTPUTS.items():
        python = source == "array_ops.cpp"
        target = os.path.join(build_dir, source.replace(".cpp", ".o"))
        compile_command = [
            "g++", "-std=c++17", "-O2", "-fPIC", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM",
            f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
            *["-I" + path for path in includes + ([sysconfig.get_paths()["include"]] if python else [])],
            "-c", os.path.join(HERE, source), "-o", target,
        ]  # fmt: skip
        link_command = [
            "g++", "-shared", "-o", output, target, "-L" + LIBRARY_DIR, "-lmops", "-L" + torch_lib,
            *(["-ltorch_python"] if python else []), "-ltorch", "-ltorch_cpu", "-ltorch_hip", "-lc10", "-lc10_hip",
            "-L" + os.path.join(rocm, "lib"), "-lamdhip64", "-Wl,-rpath,$ORIGIN", "-Wl,-rpath," + torch_lib,
            # (the interpreter itself holds the Python symbols)
            *([] if python else ["-Wl,--no-undefined"]),
        ]  # fmt: skip
        process = subprocess.Popen(compile_command, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
        running.append((process, compile_command, link_command))
    for process, compile_command, link_command in running:
        log, _ = process.communicate()
        if process.returncode != 0:
            raise RuntimeError(f"{' '.join(compile_command)} failed:\n{log[-4000:]}")
        done = subprocess.run(link_command, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
        if done.returncode != 0:
            raise RuntimeError(f"{' '.join(link_command)} failed:\n{done.stdout[-4000:]}")
    return list(OUTPUTS.values())


if __name__ == "__main__":
    print("built", *build())
    sys.exit(0)
