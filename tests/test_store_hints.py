"""The reconstruction kernels hold their output stores in two forms, past the
caches and through them.  The hint is metadata to the compiler, which may join
the two into plain stores without a change in any result: so the machine code
that this repository's build made is looked at for both."""
import os
import re
import subprocess

import pytest

LLVM = "/opt/rocm/llvm/bin"
TOOLS = [os.path.join(LLVM, t) for t in ("llvm-objcopy", "clang-offload-bundler", "llvm-objdump")]


@pytest.fixture(scope="module")
def stores(tmp_path_factory):
    """Kernel name -> numbers of its 4- and 8-byte stores, plain and with the hint."""
    if not all(os.path.exists(t) for t in TOOLS):
        pytest.skip("no LLVM tools")
    from prism_amd import _lib
    _lib.lib()
    tmp = tmp_path_factory.mktemp("code")
    obj = os.path.join(os.path.dirname(_lib.__file__), "_build", "predictor.o")
    if not os.path.exists(obj):
        obj = os.path.join(os.path.dirname(_lib.__file__), "_build", "libprism_amd.so")
    fat = tmp / "fat"
    subprocess.run([TOOLS[0], "--dump-section", f".hip_fatbin={fat}", obj, str(tmp / "rest")], check=True)
    data = fat.read_bytes()
    at = [m.start() for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data)] + [len(data)]
    found = {}
    for i, (a, b) in enumerate(zip(at, at[1:])):
        bundle, code = tmp / f"bundle{i}", tmp / f"code{i}"
        bundle.write_bytes(data[a:b])
        subprocess.run([TOOLS[1], "--type=o", "--unbundle", f"--input={bundle}", f"--output={code}",
                        "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"], check=True)
        text = subprocess.run([TOOLS[2], "-d", "--demangle", "--no-show-raw-insn", str(code)], check=True,
                              capture_output=True, text=True).stdout
        for part in re.split(r"^[0-9a-f]+ <", text, flags=re.M)[1:]:
            name, body = part.split("\n", 1)
            s = re.findall(r"\b(?:global|flat)_store_dword(?:x2)?\b.*", body)
            found[name] = (sum(" nt" not in x for x in s), sum(" nt" in x for x in s))
    return found


# (1: decompression.)  A tile's column is 16 stores in each of a kernel's 12 bodies
# (interior or not, three code sources, two forms of round); a plane's points are 4,
# a line's 16.
@pytest.mark.parametrize("kernel,least,both", [
    ("spline_kernel<float, 1, 2>", 192, True),
    ("spline_kernel<float, 1, 1>", 192, True),
    ("spline_kernel<double, 1, 1>", 192, True),
    ("plane_kernel<float, 1>", 4, True),
    ("plane_kernel<double, 1>", 4, True),
    ("line_kernel<float, 1>", 16, False),
    ("line_kernel<double, 1>", 16, False),
    ("retr_spline_kernel<float, 2>", 192 + 4, True),
    ("retr_spline_kernel<float, 1>", 192 + 4, True),
    ("retr_spline_kernel<double, 1>", 192 + 4, True),
])
def test_both_forms_are_there(stores, kernel, least, both):
    names = [n for n in stores if "::" + kernel + "(" in n]
    assert len(names) == 1, (kernel, sorted(stores)[:40])
    plain, hinted = stores[names[0]]
    print(kernel, "plain", plain, "past the caches", hinted)
    assert hinted >= least
    assert plain >= least if both else plain == 0
