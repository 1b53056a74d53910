"""Every global and LDS address of the kernels, on the CPU.

The kernel sources are compiled for the host against tests/host_kernels (threads
run one after another, AddressSanitizer watches buffers of exactly the documented
extents and every LDS array) and called over random sizes, odd and ragged ones and
small devices' dispatch among them.  No kernel's global addresses depend on data
beyond clamped table and token indices, so a clean run covers the GPU's accesses
at these sizes."""
import concurrent.futures
import glob
import os
import re
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(HERE)
CSRC = os.path.join(REPO, "mamba-integer_amd", "csrc")
HOST = os.path.join(HERE, "host_kernels")
UNITS = ["bitlinear", "block", "common", "decode", "mfma_scan", "model_scan", "scan"]

_SAT = "{ const int64_t q = (int64_t)%s * %s + d; r = (int)(q > INT32_MAX ? INT32_MAX : q < INT32_MIN ? INT32_MIN : q); }"


def _clang():
    for c in ("/opt/rocm/lib/llvm/bin/clang++", "/opt/rocm/llvm/bin/clang++"):
        if os.path.exists(c):
            return c
    return shutil.which("clang++")


def _host_source(text):
    """The source with its inline assembly in C and dynamic LDS as an exact allocation."""
    text = re.sub(r'asm\("v_mad_i32_i24[^;]*;', _SAT % ("b", "x"), text)
    text = re.sub(r'asm\("v_mad_i32_i16 [^;"]*op_sel[^;]*;', _SAT % ("(bw >> 16)", "(xw >> 16)") , text)
    text = re.sub(r'asm\("v_mad_i32_i16 [^;]*;', _SAT % ("(int16_t)bw", "(int16_t)xw"), text)
    text = re.sub(r'\basm( volatile)?\("(s_waitcnt[^"]*)?" *:[^;]*;', ";", text)
    text = re.sub(r"extern __shared__ __align__\(16\) int8_t smem\[\];", "int8_t *smem = host_dynamic_lds;", text)
    assert not re.search(r"^[^/\n]*\basm\b *(volatile)? *\(", text, re.M), "inline assembly without a host form"
    return text


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    clang = _clang()
    if clang is None:
        pytest.skip("no clang++")
    tmp = tmp_path_factory.mktemp("host_kernels")
    for f in glob.glob(os.path.join(CSRC, "*.hpp")) + [os.path.join(CSRC, u + ".hip") for u in UNITS]:
        with open(f) as src, open(tmp / os.path.basename(f).replace(".hip", ".cpp"), "w") as dst:
            dst.write(_host_source(src.read()))
    shutil.copy(os.path.join(HOST, "addresses.cpp"), tmp)
    flags = ["-std=c++17", "-O1", "-g", "-w", "-fno-strict-aliasing", "-fsanitize=address", f"-I{HOST}", f"-I{tmp}",
             f"-I{os.path.join(REPO, 'include')}"]

    def compile_one(unit):
        out = subprocess.run([clang, *flags, "-c", str(tmp / (unit + ".cpp")), "-o", str(tmp / (unit + ".o"))],
                             capture_output=True, text=True)
        assert out.returncode == 0, out.stderr[:3000]

    units = UNITS + ["addresses"]
    with concurrent.futures.ThreadPoolExecutor(max_workers=min(8, os.cpu_count() or 1)) as pool:
        list(pool.map(compile_one, units))
    exe = tmp / "addresses"
    out = subprocess.run([clang, "-fsanitize=address", *[str(tmp / (u + ".o")) for u in units], "-o", str(exe)],
                         capture_output=True, text=True)
    assert out.returncode == 0, out.stderr[:3000]
    return str(exe)


@pytest.mark.parametrize("family,count", [("bitlinear", 120), ("bitlinear_f32", 60), ("block", 50), ("block_2103", 1),
                                          ("ssd_scan", 50), ("scans", 40), ("elementwise", 60), ("decode", 30),
                                          ("limits", 0)])
def test_addresses_in_bounds(program, family, count):
    out = subprocess.run([program, family, str(count), "1"], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, (out.stdout + out.stderr)[-6000:]
