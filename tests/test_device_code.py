"""CPU checks of the device code as the library's own flags compile it."""
import os
import re
import shlex
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "infer_train_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def _device_ir(name, tmp_path):
    """{kernel: lines} of a source's optimised device IR."""
    if not (os.path.exists(HIPCC) and shutil.which("make")):
        pytest.skip("hipcc or make not found")
    obj = os.path.join(str(tmp_path), name + ".o")
    out = subprocess.run(["make", "-n", "-B", "-C", CSRC, f"BUILD={tmp_path}", obj], capture_output=True, text=True, check=True).stdout
    cmd = next(shlex.split(line) for line in out.splitlines() if name + ".hip" in line)
    ll = os.path.join(str(tmp_path), name + ".ll")
    cmd[cmd.index("-c"):] = ["--cuda-device-only", "-S", "-emit-llvm", os.path.join(CSRC, name + ".hip"), "-o", ll]
    subprocess.run(cmd, check=True, capture_output=True, timeout=300)
    kernels, body = {}, None
    for line in open(ll):
        m = re.match(r"define .*amdgpu_kernel .*@(\w+)\(", line)
        if m:
            body = kernels[m.group(1)] = []
        elif line.startswith("}"):
            body = None
        elif body is not None:
            body.append(line)
    return kernels


def _unordered(lines):
    """LDS accesses that a path reaches from one of the other kind (load after
    store, store after load) with no wavefront fence between."""
    blocks, at = {"entry": []}, "entry"
    for line in lines:
        m = re.match(r"([\w.$-]+):", line)
        if m:
            at = m.group(1)
            blocks[at] = []
        else:
            blocks[at].append(line)
    bad = set()
    reach = {b: set() for b in blocks}  # kinds that may be unfenced at the block's start
    todo = ["entry"]
    seen = set()
    while todo:
        b = todo.pop()
        seen.add(b)
        open_kinds = set(reach[b])
        for line in blocks[b]:
            if "fence syncscope(\"wavefront\")" in line:
                open_kinds.clear()
            m = re.search(r"\b(load|store) .*ptr addrspace\(3\)", line)
            if m:
                if open_kinds - {m.group(1)}:
                    bad.add(line.strip())
                open_kinds.add(m.group(1))
        for nxt in re.findall(r"label %([\w.$-]+)", "".join(blocks[b])):
            if nxt not in seen or not open_kinds <= reach[nxt]:
                reach[nxt] |= open_kinds
                todo.append(nxt)
    return sorted(bad)


def test_wave_private_lds_stages_are_fenced(tmp_path):
    """The quantised append and gather hand bytes from lane to lane through a
    wave-private LDS stage, written and read as different types and at
    different addresses of a lane: only a fence keeps the compiler from moving
    the reads before the writes (or the next chunk's writes before the
    reads)."""
    kernels = _device_ir("it_cache", tmp_path)
    staged = {k: v for k, v in kernels.items() if any("ptr addrspace(3)" in line for line in v)}
    names = "".join(staged)
    assert all(n in names for n in ("kv_append_q8_wide", "kv_append_nib_wide", "kv_gather_quant"))
    bad = {k: b for k, b in ((k, _unordered(v)) for k, v in staged.items()) if b}
    assert not bad, {k: b[:3] for k, b in bad.items()}


def _kernel_registers():
    """{kernel: (VGPRs, spilled VGPRs)} of the built library's code objects."""
    import struct

    from infer_train_amd._lib import LIB_PATH

    readelf = "/opt/rocm/llvm/bin/llvm-readelf"
    if not os.path.exists(readelf):
        pytest.skip("llvm-readelf not found")
    data = open(LIB_PATH, "rb").read()
    magic, found, at = b"__CLANG_OFFLOAD_BUNDLE__", {}, 0
    while (at := data.find(magic, at)) >= 0:
        p = at + len(magic) + 8
        for _ in range(struct.unpack_from("<Q", data, p - 8)[0]):
            off, size, n = struct.unpack_from("<QQQ", data, p)
            if b"gfx950" in data[p + 24:p + 24 + n] and size:
                notes = subprocess.run([readelf, "--notes", "-"], input=data[at + off:at + off + size], capture_output=True,
                                       check=True).stdout.decode()
                for block in notes.split(".agpr_count:")[1:]:
                    name, v, s = (re.search(rf"\.{key}:\s+(\S+)", block) for key in ("name", "vgpr_count", "vgpr_spill_count"))
                    found[name[1]] = int(v[1]), int(s[1])
            p += 24 + n
        at += len(magic)
    return found


def test_decode_registers_allow_the_planned_waves():
    """The partition planner counts on the waves that a SIMD's 512 VGPRs hold
    (allocated in eights) of the quantised decode at head_dim 128 in two-wave
    workgroups: four, three for four of Q5_1's head counts; none of them spills."""
    from infer_train_amd import _lib as L

    regs, seen = _kernel_registers(), 0
    for name, (vgprs, spilled) in regs.items():
        m = re.search(r"paged_decode_splitILi(\d+)ELi128ELi(\d+)ELi2ELi2E", name)
        if not m or int(m[1]) not in (L.Q4_0, L.Q4_1, L.Q5_0, L.Q5_1, L.Q8_0):
            continue
        seen += 1
        want = 3 if int(m[1]) == L.Q5_1 and int(m[2]) in (2, 5, 6, 7) else 4
        assert 512 // (-(-vgprs // 8) * 8) >= want and spilled == 0, (name, vgprs, spilled)
    assert seen == 5 * 8  # formats, head counts


_QUANT_CODE = r"""
#include <cmath>
#include <cstdio>
#include "it_device.hpp"
#include "it_quant.hpp"
using namespace itkv;
int main() {
  const float inf = INFINITY, r[] = {0.0f, -0.0f, 0.49f, 0.999f, 1.0f, 8.5f, 15.99f, 16.0f, 31.5f, 32.99f, inf, -inf, NAN, -NAN};
  const unsigned want[] = {0, 0, 0, 0, 1, 8, 15, 16, 31, 32, 0, 0, 0, 0};
  for (unsigned top : {15u, 31u})
    for (int i = 0; i < 14; ++i) {
      const unsigned w = want[i] < top ? want[i] : top;
      if (quant_code(r[i], top) != w) return printf("%g: %u, not %u\n", double(r[i]), quant_code(r[i], top), w), 1;
    }
  return 0;
}
"""


def test_quant_code_is_defined_for_every_value(tmp_path):
    """quant_code on the host, with conversions out of range trapped: the
    infinities of an overflowed 1 / d have the code 0 of a NaN."""
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not found")
    src, exe = tmp_path / "code.hip", str(tmp_path / "code")
    src.write_text(_QUANT_CODE)
    cmd = [HIPCC, "--offload-arch=gfx950", "-std=c++17", "-O1", "-I", CSRC, "-I", os.path.join(ROOT, "include"),
           "-Xarch_host", "-fsanitize=float-cast-overflow", "-Xarch_host", "-fsanitize-trap=all", str(src), "-o", exe]
    b = subprocess.run(cmd, capture_output=True, text=True, timeout=300)
    assert b.returncode == 0, b.stderr[-2000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout)


def test_profiled_kernels_exist():
    """The kernels that the profile summaries look for are in the library: the
    movers' by name, the instruction census's exactly one each."""
    import bench

    names = list(_kernel_registers())
    for workload, kernel, *_ in bench.movers_plan():
        base, _, arg = kernel.partition("<")
        symbol = base + (f"ILi{arg}E" if arg else "")
        assert any(symbol in n for n in names), workload
    for _, symbol, _ in bench.ISA_KERNELS:
        assert sum(symbol in n for n in names) == 1, symbol
