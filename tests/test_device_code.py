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
