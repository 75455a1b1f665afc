"""Builds the native library libcombustion_amd.so in place (host C++ against the HIP runtime and hiprtc).

The mechanism-specialised gfx950 kernels are generated and compiled at assemble time by hiprtc (or ahead of
time into the code-object cache by `precompile`). Usage: python -m combustion_amd.build
"""
import os
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libcombustion_amd.so")
TENSORS = os.path.join(HERE, "_tensors.so")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
SOURCES = ["yaml.cpp", "mechanism.cpp", "ast.cpp", "reaction.cpp", "transport.cpp", "hip_emit.cpp", "device.cpp",
           "forms.cpp", "rates_split.cpp", "transport_split.cpp", "tiled.cpp", "mlp.cpp", "export.cpp", "ignition.cpp", "host_jit.cpp", "jacobian.cpp", "integrator.cpp", "capi.cpp"]


KERNELS = {"rates_mixed_source": "rates_mixed.hip", "transport_tiled_source": "transport_tiled.hip",
           "mlp_source": "mlp.hip", "rosenbrock_source": "rosenbrock.hip", "rates_tiled_source": "rates_tiled.hip",
           "surrogate_source": "surrogate.hip", "rates_split_source": "rates_split.hip",
           "transport_split_source": "transport_split.hip",
           "transport_pairs_source": "transport_pairs.hip"}


def embed_kernels():
    """Writes _build/embedded_kernels.cpp holding the HIP kernel templates as strings."""
    out = ['// Generated by combustion_amd/build.py from csrc/kernels/*.hip.', 'namespace combustion {']
    for name, fn in KERNELS.items():
        with open(os.path.join(CSRC, "kernels", fn)) as f:
            text = f.read()
        out.append(f'extern const char* const {name} = R"HIPSRC({text})HIPSRC";')
    out.append('}')
    path = os.path.join(HERE, "_build", "embedded_kernels.cpp")
    with open(path, "w") as f:
        f.write("\n".join(out) + "\n")
    return path


# Translation units with device code of their own (compiled by hipcc for gfx950; the HIP runtime registers their
# code objects when the library loads).
HIP_SOURCES = ["noalloc.hip"]


def build_tensors():
    """Starts the compilation of the torch tensor helper (csrc/tensors.cpp) where torch is installed."""
    try:
        import torch
        from torch.utils.cpp_extension import include_paths
    except ImportError:
        return None
    libs = os.path.join(os.path.dirname(torch.__file__), "lib")
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}"]
    cmd += ["-isystem" + d for d in include_paths() + [sysconfig.get_paths()["include"]]]
    cmd += [os.path.join(CSRC, "tensors.cpp"), "-o", TENSORS + ".tmp", "-L" + libs, "-Wl,-rpath," + libs, "-ltorch_python", "-ltorch_cpu", "-lc10"]
    return "tensors.cpp", subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)


def build(verbose=True):
    objs = []
    os.makedirs(os.path.join(HERE, "_build"), exist_ok=True)
    embedded = embed_kernels()
    procs = []
    for src in HIP_SOURCES:
        obj = os.path.join(HERE, "_build", os.path.basename(src).replace(".hip", ".hip.o"))
        cmd = [os.path.join(ROCM, "bin", "hipcc"), "-O2", "-std=c++17", "-fPIC", "--offload-arch=gfx950", "-Xclang", "-target-feature",
               "-Xclang", "-packed-fp32-ops", "-Wall", "-Wno-unused-command-line-argument", "-c", os.path.join(CSRC, src), "-o", obj]
        procs.append((src, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)))
        objs.append(obj)
    for src in SOURCES + [embedded]:
        obj = os.path.join(HERE, "_build", os.path.basename(src).replace(".cpp", ".o"))
        cmd = ["g++", "-O2", "-g", "-std=c++17", "-fPIC", "-Wall", "-Wno-unused-function", "-D__HIP_PLATFORM_AMD__",
               "-I" + os.path.join(ROCM, "include"), "-c", os.path.join(CSRC, src), "-o", obj]
        procs.append((src, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)))
        objs.append(obj)
    tensors = build_tensors()
    if tensors:
        procs.append(tensors)
    failed = False
    for src, p in procs:
        out, _ = p.communicate()
        # hipcc's host pass does not know the packed-fp32 feature flag of the device pass: that warning is expected
        out = "\n".join(l for l in (out or "").splitlines() if "packed-fp32-ops" not in l and "not a recognized feature" not in l
                        and l.strip() != "1 warning generated.")
        if out and verbose:
            sys.stdout.write(out + "\n")
        if p.returncode:
            failed = True
            sys.stdout.write(f"compile failed: {src}\n")
    if failed:
        raise RuntimeError("native build failed")
    tmp = LIB + ".tmp"
    cmd = ["g++", "-shared", "-o", tmp] + objs + ["-L" + os.path.join(ROCM, "lib"), "-Wl,-rpath," + os.path.join(ROCM, "lib"),
                                                  "-lamdhip64", "-lhiprtc", "-ldl"]
    subprocess.check_call(cmd)
    os.replace(tmp, LIB)
    if tensors:
        os.replace(TENSORS + ".tmp", TENSORS)
    return LIB


if __name__ == "__main__":
    print(build())
