"""Device-memory bookkeeping of the host layer, on the CPU: its C sources linked with a stand-in for the HIP allocator
that has 64 MB (tests/host_memory/main.c) and with empty kernels.  Storage that freed states leave behind is kept for the
next request; every other allocation of the library must still get it when the device has nothing else."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "orkan_amd", "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
GCC = shutil.which("gcc")

pytestmark = pytest.mark.skipif(GCC is None or not os.path.isdir(os.path.join(ROCM, "include", "hip")),
                                reason="needs gcc and the HIP headers")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    """the host layer, main.c, and a stub returning 0 for every function neither defines"""
    out = tmp_path_factory.mktemp("host_memory")
    srcs = [os.path.join(CSRC, f) for f in sorted(os.listdir(CSRC)) if f.endswith(".c")]
    srcs.append(os.path.join(ROOT, "tests", "host_memory", "main.c"))
    flags = ["-std=gnu17", "-O1", "-g", "-w", "-DLOG_TILE_DIM=5", "-D__HIP_PLATFORM_AMD__", "-I", CSRC, "-I",
             os.path.join(ROOT, "include"), "-I", os.path.join(ROCM, "include")]
    objs = []
    for s in srcs:
        objs.append(str(out / (os.path.basename(s) + ".o")))
        subprocess.run([GCC, *flags, "-c", s, "-o", objs[-1]], check=True)
    link = [GCC, *objs, "-o", str(out / "host_memory"), "-lm", "-lpthread"]
    r = subprocess.run(link, capture_output=True, text=True)
    missing = sorted(set(re.findall(r"undefined reference to `((?:ork_|hip)\w+)'", r.stderr)))
    assert missing, r.stderr[-2000:]
    stub = out / "stubs.c"
    stub.write_text("".join(f"long {m}() {{ return 0; }}\n" for m in missing))
    subprocess.run([GCC, "-std=gnu17", "-w", "-c", str(stub), "-o", str(out / "stubs.o")], check=True)
    subprocess.run([*link, str(out / "stubs.o")], check=True)
    return str(out / "host_memory")


def run(program, what):
    r = subprocess.run([program, what], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and f"host_memory ok {what}" in r.stdout, (r.returncode, r.stderr)


@pytest.mark.parametrize("what", ["dev_alloc", "staging", "phases", "mlp", "qaoa"])
def test_kept_storage_goes_back_when_the_device_runs_out(program, what):
    run(program, what)


@pytest.mark.parametrize("what", ["count", "classes", "cap", "behind"])
def test_what_is_kept(program, what):
    """By pages and by number, by size, at most 8 GB, and with an address freed behind the library's back."""
    run(program, what)


def test_kept_storage_is_released_on_request(program):
    run(program, "trim")


def test_batched_qaoa_scratch_is_that_of_the_configuration(program):
    run(program, "qaoa_scratch")


def test_refused_search_changes_nothing(program):
    run(program, "qaoa_refused")


def test_network_holds_each_gradient_once(program):
    """Gradients of the pre-activations take the place of activations that the backward pass is done with."""
    run(program, "mlp_size")
