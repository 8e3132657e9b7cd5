"""Static checks of the gfx950 code objects -- CPU only (hipcc cross-compiles), with the flags of the
library's Makefile.

* No kernel makes a device-function call: the balanced kernel reads its arguments through the
  kernarg-segment pointer, which is only valid in the kernel body (in a called function it is
  null), and calls would also cost registers and latency in the hot loop.
* No packed-FP32 instructions are emitted (the build disables them).
* No kernel spills registers to scratch.
* The decode kernels hold nothing in AGPRs (the build keeps MFMA accumulators in VGPRs).
* M0 is written only by the direct global->LDS loads (cascade.hip's key-split prefix kernel and the
  decode body issue them from inline asm that sets M0 and declares it clobbered): every M0 reference
  is such a write, followed by the wait state and the load, so no compiler-generated code holds a
  value in M0 across them.
* The device pass prints no warning.

Every .hip source of the library is checked.
"""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "cuda-kernel-lab_amd")
CSRC = os.path.join(PKG, "csrc")
HIPCC = "/opt/rocm/bin/hipcc"
needs_hipcc = pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")


def _makefile_flags():
    """CXXFLAGS and HIPFLAGS as make expands them."""
    text = subprocess.run(["make", "-C", PKG, "-pnq", "-f", "Makefile"], capture_output=True, text=True).stdout
    value = {m.group(1): m.group(2) for m in re.finditer(r"^(CXXFLAGS|HIPFLAGS|ARCH) :?\??= (.*)$", text, re.M)}
    flags = (value["CXXFLAGS"] + " " + value["HIPFLAGS"]).replace("$(ARCH)", value["ARCH"])
    assert "$" not in flags, flags
    return flags.split()


SOURCES = sorted(f[:-4] for f in os.listdir(CSRC) if f.endswith(".hip"))


@pytest.fixture(scope="module")
def built(tmp_path_factory):
    """name -> (assembly, what the compiler said), each source compiled once."""
    cache, flags = {}, _makefile_flags()

    def get(name):
        if name not in cache:
            out = tmp_path_factory.mktemp("lint") / (name + ".s")
            r = subprocess.run([HIPCC, *flags, "--cuda-device-only", "-S", os.path.join(CSRC, name + ".hip"), "-o",
                                str(out), "-Rpass-analysis=kernel-resource-usage"],
                               check=True, capture_output=True, text=True)
            cache[name] = out.read_text(), r.stderr
        return cache[name]
    return get


def test_every_source_is_linted():
    assert {"decode", "cascade", "append", "misc", "noalloc"} <= set(SOURCES)


@needs_hipcc
def test_the_lint_builds_what_ships():
    flags = " ".join(_makefile_flags())
    for f in ("-O3", "--offload-arch=gfx950", "-Xclang -target-feature -Xclang -packed-fp32-ops",
              "-mllvm -amdgpu-mfma-vgpr-form"):
        assert f in flags, f


@needs_hipcc
@pytest.mark.parametrize("name", SOURCES)
def test_no_calls_no_packed_fp32(name, built):
    asm, _ = built(name)
    assert "s_swappc_b64" not in asm, f"{name}.hip: a kernel calls a device function"
    assert not re.search(r"\bv_pk_(add|mul|fma)_f32\b", asm), f"{name}.hip: packed FP32 emitted"


@needs_hipcc
@pytest.mark.parametrize("name", SOURCES)
def test_no_scratch_spills(name, built):
    _, text = built(name)
    names = re.findall(r"Function Name: (\S+)", text)
    spills = re.findall(r"VGPRs Spill: (\d+)", text)
    sspills = re.findall(r"SGPRs Spill: (\d+)", text)
    scratch = re.findall(r"ScratchSize \[bytes/lane\]: (\d+)", text)
    assert len(names) == len(spills) == len(sspills) == len(scratch)
    if name != "noalloc":   # (noalloc.hip holds a device array and host code, no kernel)
        assert names
    for n, sp, ss, sc in zip(names, spills, sspills, scratch):
        assert int(sp) == 0 and int(ss) == 0, f"{name}.hip: {n} spills {sp} VGPRs, {ss} SGPRs"
        assert int(sc) == 0, f"{name}.hip: {n} uses {sc} bytes of scratch"


@needs_hipcc
def test_decode_accumulators_are_in_vgprs(built):
    _, text = built("decode")
    agprs = dict(zip(re.findall(r"Function Name: (\S+)", text), re.findall(r" AGPRs: (\d+)", text)))
    assert agprs and all(int(a) == 0 for a in agprs.values()), agprs


@needs_hipcc
@pytest.mark.parametrize("name", SOURCES)
def test_no_warnings(name, built):
    _, text = built(name)
    said = [ln for ln in text.splitlines() if "warning:" in ln and not ln.startswith("clang")]   # (not the driver's)
    assert not said, said[:5]


@needs_hipcc
@pytest.mark.parametrize("name", SOURCES)
def test_m0_only_for_direct_lds_loads(name, built):
    asm, _ = built(name)
    lines = [ln.split(";")[0].strip() for ln in asm.splitlines()]
    lines = [ln for ln in lines if ln]
    uses = [i for i, ln in enumerate(lines) if re.search(r"\bm0\b", ln)]
    loads = sum(1 for ln in lines if ln.startswith("global_load_lds_dwordx4"))
    assert len(uses) == loads
    assert bool(uses) == (name in ("cascade", "decode"))
    for i in uses:
        assert re.fullmatch(r"s_mov_b32 m0, s\d+", lines[i]), lines[i]
        assert lines[i + 1] == "s_nop 0" and lines[i + 2].startswith("global_load_lds_dwordx4"), lines[i:i + 3]
