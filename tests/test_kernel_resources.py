"""The kernels' register / LDS budget, read from the compiler's resource report (no GPU needed: hipcc cross-compiles).
The design leans on it: a spill reload inside the key loop is a vector load that drains the whole tile queue, any scratch
at all costs a launch about 0.7 us, and the single-buffered build only pays if two of its workgroups fit a CU (half the
register file, 80 KB of LDS)."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "p100e-engine_amd", "csrc")


def resource_report(tmp_path, source="p1a_decode.hip", flags=()):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc here")
    cmd = [hipcc, "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-I" + os.path.join(ROOT, "include"), "-I" + SRC,
           "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-Wno-unused-command-line-argument", "-Wno-inline-asm",
           "-Rpass-analysis=kernel-resource-usage", "--cuda-device-only", *flags, "-c", os.path.join(SRC, source), "-o", str(tmp_path / "out.o")]
    r = subprocess.run(cmd, capture_output=True, text=True, timeout=900)
    assert r.returncode == 0, r.stderr[-2000:]
    kernels, cur = {}, None
    for line in r.stderr.splitlines():
        m = re.search(r"Function Name: (\S+)", line)
        if m:
            cur = kernels.setdefault(m.group(1), {})
            continue
        m = re.search(r"remark:\s+([A-Za-z ]+?)(?: \[[^\]]*\])?: (\d+)", line)
        if m and cur is not None:
            cur[m.group(1).strip()] = int(m.group(2))
    return kernels


def test_decode_kernels_fit_their_budget(tmp_path):
    ks = {k: v for k, v in resource_report(tmp_path).items() if "dec_mfma_k" in k}
    assert len(ks) >= 12, sorted(ks)
    for name, r in ks.items():
        assert r.get("VGPRs Spill", 0) == 0 and r.get("SGPRs Spill", 0) == 0, (name, r)
        assert r.get("ScratchSize", 0) == 0, (name, r)
    # dec_mfma_k<KT, D, NT, NW, SB, KS>: the mangled name ends ...ELi<NW>ELb<SB>ELj<KS>EEEv...
    sb = {k: v for k, v in ks.items() if re.search(r"ELb1ELj\d+EEEv", k)}
    assert len(sb) >= 5, sorted(ks)
    # the staged builds (KS != KT: q8_0 / q4_0 at D = 64, 128 converted to f16 tiles) are there, one workgroup per CU
    staged = {k: v for k, v in ks.items() if re.search(r"ILj1ELi(64|128)ELi[12]ELi8ELb0ELj[28]EEEv", k)}
    assert len(staged) == 8, sorted(ks)
    for name, r in staged.items():
        assert r["LDS Size"] <= 160 * 1024, (name, r)
    for name, r in sb.items():
        waves = int(re.search(r"ELi(\d+)ELb1ELj\d+EEEv", name).group(1))
        assert r["LDS Size"] <= 80 * 1024, (name, r)                       # two workgroups in 160 KB
        assert r["Occupancy"] * 4 >= 2 * waves, (name, r)                   # two workgroups' waves on the 4 SIMDs


LIST, LOOP, DIRECT = 256, 512, 1024                            # what the last argument holds beside the cache's type


def builds(names):
    """dec_mfma_k<KT, D, NT, NWV, SB, HOW> by mangled name: its arguments, HOW taken apart as the cache's type and the kind of build"""
    out = {}
    for name in names:
        kt, D, nt, nwv, sb, how = (int(x) for x in re.search(r"dec_mfma_kILj(\d+)ELi(\d+)ELi(\d+)ELi(\d+)ELb([01])ELj(\d+)EEEv", name).groups())
        assert not how & ~(255 | LIST | LOOP | DIRECT), name
        out[name] = {"D": D, "NT": nt, "waves": nwv, "sb": sb, "staged": how & 255 != kt, "kind": how & ~255}
    return out


def test_every_kind_of_decode_build_fits_its_budget(tmp_path):
    """the builds for a stream a workgroup, for calls of several sequences - a list of streams, one a workgroup (every build) and several (the single-buffered and the
    staged ones, two column tiles of f16 and q8_0) - and for calls of one unit, each with the double-buffered, single-buffered and staged builds it has: none spills, and two
    workgroups of a single-buffered one fit a CU, staged or not"""
    ks = {k: v for k, v in resource_report(tmp_path).items() if "dec_mfma_k" in k}
    of = builds(ks)
    counts = {}
    for b in of.values():
        key = (b["kind"], b["sb"], b["staged"])
        counts[key] = counts.get(key, 0) + 1
    assert counts == {(0, 0, False): 10, (0, 0, True): 8, (0, 1, False): 5, (0, 1, True): 2,
                      (LIST, 0, False): 10, (LIST, 0, True): 8, (LIST, 1, False): 5, (LIST, 1, True): 2,
                      (LIST | LOOP, 0, False): 4, (LIST | LOOP, 0, True): 8, (LIST | LOOP, 1, False): 5, (LIST | LOOP, 1, True): 2,
                      (DIRECT, 0, False): 9, (DIRECT, 0, True): 8}
    for name, r in ks.items():
        assert all(r.get(x, 0) == 0 for x in ("VGPRs Spill", "SGPRs Spill", "ScratchSize")), (name, r)
        two = of[name]["sb"]
        assert r["LDS Size"] <= (80 if two else 160) * 1024, (name, r)
        assert r["Occupancy"] * 4 >= (2 if two else 1) * of[name]["waves"], (name, r)


def test_decode_kernels_make_no_flat_access(tmp_path):
    """tiles are waited for by count; a FLAT access in flight (a pointer the compiler does not know to be one to device memory) leaves
    only the wait for everything defined"""
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc here")
    out = tmp_path / "decode.s"
    r = subprocess.run([hipcc, "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-I" + os.path.join(ROOT, "include"), "-Xclang", "-target-feature", "-Xclang",
                        "-packed-fp32-ops", "-Wno-unused-command-line-argument", "-Wno-inline-asm", "--cuda-device-only", "-S",
                        os.path.join(SRC, "p1a_decode.hip"), "-o", str(out)], capture_output=True, text=True, timeout=900)
    assert r.returncode == 0, r.stderr[-2000:]
    kernel, flat, seen = "", set(), set()
    for line in out.read_text().splitlines():
        m = re.match(r"(_ZN\S*dec_mfma_k\S*):", line)
        if m or re.match(r"\S+:", line) and not line.startswith("."):
            kernel = m.group(1) if m else ""
        if kernel:
            seen.add(kernel)
            if re.match(r"\s+flat_", line):
                flat.add(kernel)
    assert len(seen) >= 40 and not flat, (len(seen), sorted(flat))


VGPR_FORM = ("-mllvm", "-amdgpu-mfma-vgpr-form")               # (as the Makefile builds these two)


def test_prefill_kernels_fit_their_budget(tmp_path):
    """one workgroup of four waves to a CU, two where D <= 128 and the tiles come straight into LDS; nothing in memory. Scalar
    registers do spill, to lanes of vector registers (reading the arguments again behind the key loop takes all of that out
    and costs 0.3 us a call): not more than they do"""
    ks = {k: v for k, v in resource_report(tmp_path, "p1a_prefill.hip", VGPR_FORM).items() if "prefill_k" in k}
    assert len(ks) == 21, sorted(ks)
    for name, r in ks.items():                                 # prefill_k<KT, D, GROUPED, DMA>
        D, dma = int(re.search(r"ELi(\d+)ELb", name).group(1)), "ELb1ELb1E" in name
        assert r.get("VGPRs Spill", 0) == 0 and r.get("ScratchSize", 0) == 0, (name, r)
        assert r.get("SGPRs Spill", 0) <= (2 if dma else 19), (name, r)
        assert r["Occupancy"] >= (2 if dma and D <= 128 else 1), (name, r)


def test_any_shape_kernels_fit_their_budget(tmp_path):
    """a build for each of 16 head sizes and three types, none of which spills; up to 256 dims eight waves, two to a SIMD, and LDS
    for two workgroups on a CU"""
    ks = {k: v for k, v in resource_report(tmp_path, "p1a_decode_any.hip", VGPR_FORM).items() if "dec_any_k" in k}
    assert len(ks) == 48, sorted(ks)
    for name, r in ks.items():                                 # dec_any_k<KT, blocks of 32 dims, waves>
        blocks = int(re.search(r"ILj\d+ELi(\d+)ELi", name).group(1))
        assert all(r.get(x, 0) == 0 for x in ("VGPRs Spill", "SGPRs Spill", "ScratchSize")), (name, r)
        assert r["LDS Size"] <= 80 * 1024 and r["Occupancy"] >= (2 if blocks <= 8 else 1), (name, r)
