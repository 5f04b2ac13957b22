"""Small uploads are left to the order of a device's default stream until the block's address is handed out: kept by device, on
two devices that a stand-in runtime makes up (no GPU needed)."""
import concurrent.futures
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(ROOT, "spoc_amd", "csrc")
CLANG = "/opt/rocm/llvm/bin/clang++"


@pytest.mark.skipif(not os.path.exists(CLANG), reason="no clang++ in this image")
def test_small_uploads_are_waited_for_on_their_own_device(tmp_path):
    sources = [os.path.join(HERE, "host_sanitizers", f) for f in ("two_devices.cpp", "kernel_stubs.cpp")]
    sources += [os.path.join(CSRC, f) for f in (
        "status.cpp", "backend_info.cpp", "tunables.cpp", "runtime.cpp", "vector.cpp", "gpu_memory.cpp", "code_cache.cpp",
        "plugin.cpp", "library_kernels.cpp", "generate.cpp", "fusion_abi.cpp", "host/ir_text.cpp", "host/ir_hip.cpp",
        "host/specialise.cpp", "host/fusion.cpp", "host/map_fuse.cpp")]
    flags = ["-std=c++20", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I" + os.path.join(ROOT, "include"),
             "-I" + CSRC, "-w"]

    def compile_one(item):
        k, src = item
        obj = str(tmp_path / f"{k}.o")
        done = subprocess.run([CLANG, *flags, "-c", src, "-o", obj], capture_output=True, text=True)
        assert done.returncode == 0, done.stderr[-3000:]
        return obj
    with concurrent.futures.ThreadPoolExecutor(max_workers=8) as pool:
        objects = list(pool.map(compile_one, enumerate(sources)))
    exe = str(tmp_path / "two_devices")
    link = subprocess.run([CLANG, *objects, "-L/opt/rocm/lib", "-lamdhip64", "-lhiprtc", "-lpthread", "-Wl,-rpath,/opt/rocm/lib",
                           "-o", exe], capture_output=True, text=True)
    assert link.returncode == 0, link.stderr[-3000:]
    run = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0 and "two devices ok" in run.stdout, run.stdout + run.stderr
