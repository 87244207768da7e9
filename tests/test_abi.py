"""CPU checks of the C ABI: the library loads without a GPU, exports every
function include/it_kv.h declares, and validates arguments before touching
the device (no compute is launched here)."""
import ctypes as C
import os
import re

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared():
    src = open(os.path.join(ROOT, "include", "it_kv.h")).read()
    src = re.sub(r"/\*.*?\*/", "", src, flags=re.S)
    return sorted(set(re.findall(r"\b(it_[a-z0-9_]+)\s*\(", src)))


def test_every_declared_symbol_is_exported():
    from infer_train_amd._lib import LIB_PATH, SIGNATURES

    raw = C.CDLL(LIB_PATH)
    names = _declared()
    assert len(names) >= 35
    missing = [n for n in names if not hasattr(raw, n)]
    assert not missing, missing
    assert set(names) == set(SIGNATURES), set(names) ^ set(SIGNATURES)


def test_product_does_not_reference_oracle():
    pkg = os.path.join(ROOT, "infer_train_amd")
    for dirpath, _, files in os.walk(pkg):
        for f in files:
            if f.endswith((".py", ".hip", ".cpp", ".hpp", ".h", "Makefile")):
                text = open(os.path.join(dirpath, f), errors="replace").read()
                assert "import oracle" not in text and "liboracle" not in text and "it_oracle" not in text, f


def test_status_codes_and_pure_queries():
    from infer_train_amd import _lib as L

    lib = L.lib
    assert lib.it_abi_version() == 1
    assert lib.it_supports(L.OP_PAGED_DECODE, L.BF16) == 1
    assert lib.it_supports(L.OP_PAGED_DECODE, L.Q4_0) == 1
    assert lib.it_supports(L.OP_PAGED_DECODE, L.Q4_1) == 1
    for dt in (L.Q5_0, L.Q5_1):
        for op in (L.OP_KV_APPEND, L.OP_KV_GATHER, L.OP_KV_EVICT, L.OP_KV_COPY_BLOCKS, L.OP_PAGED_DECODE):
            assert lib.it_supports(op, dt) == 1
        assert lib.it_supports(L.OP_PAGED_PREFILL, dt) == 0
    assert lib.it_supports(L.OP_PAGED_DECODE, 9) == 0  # Q8_1 caches are not implemented
    assert lib.it_kv_page_bytes(32, 256, L.Q4_1) == 32 * 128 + 32 * 8 * 4  # 5120
    # nibble plane + per token 8 groups of (qh u32, d fp16) / (qh u32, d and m fp16)
    assert lib.it_kv_page_bytes(16, 128, L.Q5_0) == 16 * 64 + 16 * 4 * 6  # 1408 = 16 x 4 x 22 bytes
    assert lib.it_kv_page_bytes(32, 256, L.Q5_1) == 32 * 128 + 32 * 8 * 8  # 6144 = 32 x 8 x 24 bytes
    assert lib.it_supports(L.OP_PAGED_PREFILL, L.Q4_0) == 0
    assert lib.it_supports(L.OP_PAGED_PREFILL, L.BF16) == 1
    assert lib.it_supports(L.OP_PAGED_PREFILL, L.F16) == 1  # F16 caches run the same MFMA kernel
    assert lib.it_kv_page_bytes(32, 256, L.Q4_0) == 32 * 128 + 32 * 8 * 2  # 4608
    assert lib.it_kv_page_bytes(16, 128, L.BF16) == 4096
    assert lib.it_kv_page_bytes(32, 256, L.Q8_0) == 32 * 256 + 32 * 8 * 2  # 8704
    assert lib.it_kv_page_bytes(16, 128, L.F32) == 8192
    ws = lib.it_paged_decode_workspace(32, 28, 128, 4097, 512)
    assert ws >= 32 * 28 * 9 * (128 + 2) * 4


def test_decode_partition_planner():
    """it_paged_decode_partition: the smallest multiple of 64 whose
    non-empty units run in the fewest rounds of four resident workgroups per
    compute unit (host arithmetic, no device with n_cu given)."""
    import numpy as np

    from infer_train_amd import _lib as L
    from infer_train_amd.kv import decode_partition

    def plan(ctx, start=None, hq=28, hkv=4, dt=L.BF16, D=128, bs=16, n_cu=256):
        return decode_partition(dt, D, bs, hq, hkv, ctx, start, n_cu)

    # Config 2 at 4k: 32 x 4 heads x 8 partitions of 512 = 1024 = 4 x 256.
    assert plan(np.full(32, 4096)) == 512
    # Config 2 as specified (ragged): 256-token partitions give 1024 units.
    ctx = np.random.default_rng(22).integers(256, 4097, 32) + 1
    assert plan(ctx) == 256
    units = lambda p: int(sum((c + p - 1) // p for c in ctx)) * 4
    assert units(256) <= 1024 < units(192)
    # One 1024-token sequence (config 1 heads): the shortest partition.
    assert plan([1024], hq=12, hkv=2, dt=L.F32) == 64
    # Windows count only [start, ctx); empty batches take the shortest.
    assert plan(np.full(32, 8192), np.full(32, 8192 - 4096)) == 512
    assert plan([0, 5], [0, 5]) == 64
    # Half the compute units: 512-token partitions take 2 rounds of 512
    # slots; 1024-token ones also 2 (their LDS leaves 2 per CU); shorter
    # ones 3 or more.
    assert plan(np.full(32, 4096), n_cu=128) == 512
    # Config 5 (Q8_0, D 256, block 32, 16 x U[32k, 128k]) needs many rounds
    # at any size: the longest partition with two workgroups per CU (at
    # 1792 tokens a 4-wave workgroup takes just under 80 KiB of LDS; at
    # 1856 it would not fit twice).
    c5 = np.random.default_rng(5).integers(32768, 131073, 16)
    assert plan(c5, hq=24, hkv=4, dt=L.Q8_0, D=256, bs=32) == 1792
    assert plan(c5, hq=24, hkv=4, dt=L.Q4_0, D=256, bs=32) == 1920
    with pytest.raises(L.InvalidInput):
        plan([5], hq=7, hkv=2)
    with pytest.raises(L.NotImplementedOp):
        plan([5], D=96)
    with pytest.raises(ValueError):
        plan([5, 6], [1])


def test_invalid_input_before_device():
    from infer_train_amd import _lib as L

    lib = L.lib
    assert lib.it_kv_append(None, None, None, L.BF16, None, 1, None) == L.INVALID_INPUT
    assert b"NULL" in lib.it_last_error()
    assert lib.it_kv_gather(None, None, 1, None, None, None, 1, 1, None, None, None) == L.INVALID_INPUT
    assert lib.it_paged_decode(None, None, L.BF16, 28, None, 1, None, None, 1, 1, C.c_float(0.1), 512, None, 0,
                               None, L.BF16, None) == L.INVALID_INPUT
    assert lib.it_flash_attention(None, None, None, None, None, 1, 128, 1, None, 0, None) == L.INVALID_INPUT
    h = C.c_void_p()
    assert lib.it_kv_cache_new(0, 16, 12, 2, 128, L.BF16, C.byref(h)) == L.NOT_IMPLEMENTED  # bs not 2^k
    assert lib.it_kv_cache_new(0, 16, 16, 2, 100, L.Q8_0, C.byref(h)) == L.INVALID_INPUT  # D % 32
    assert lib.it_kv_cache_new(0, 16, 16, 2, 128, 9, C.byref(h)) == L.NOT_IMPLEMENTED  # Q8_1
    assert lib.it_kv_cache_new(0, 16, 16, 2, 100, L.Q5_1, C.byref(h)) == L.INVALID_INPUT  # D % 32
    assert lib.it_kv_cache_new(0, 16, 16, 2, 96 + 8, L.Q4_0, C.byref(h)) == L.INVALID_INPUT  # D % 32


def test_python_error_mapping():
    from infer_train_amd import BlockPool, InvalidInput

    p = BlockPool(2)
    with pytest.raises(InvalidInput):
        p.free(1)


def test_decode_partition_planner_quantised_128():
    """Quantised caches at head_dim 128 run up to eight two-wave workgroups
    per compute unit (LDS permitting): partitions above 384 tokens are planned
    for that; shorter ones, and every other kernel, for four."""
    from infer_train_amd import _lib as L
    from infer_train_amd.kv import decode_partition

    def plan(ctx, hq, hkv, dt, D=128):
        return decode_partition(dt, D, 16, hq, hkv, ctx, None, 256)

    even = np.full(16, 9216)
    units = lambda p: int(sum((c + p - 1) // p for c in even)) * 8  # noqa: E731
    p = plan(even, 32, 8, L.Q4_0)
    assert p == 576 and units(p) <= 8 * 256 < units(p - 64)  # one round of eight per unit
    assert plan(even, 32, 8, L.Q8_0) == 576 and plan(even, 32, 8, L.Q5_1) == 576
    assert plan(even, 32, 8, L.BF16) == plan(even, 32, 8, L.F16)  # four per unit
    assert plan(even, 32, 8, L.BF16) != 576
    # 32 x 1024 over 4 KV heads: 128-token partitions at four per unit, kept.
    assert plan(np.full(32, 1024), 28, 4, L.Q4_0) == 128
    # Only partitions that leave room for eight (LDS is given out in pieces of 1280 bytes): not 832 tokens at
    # four of what looks like five, nor the 1984 that run in the fewest rounds of four.
    assert plan(np.full(8, 32768), 28, 4, L.Q4_0) == 256
    assert plan(np.full(9, 53787), 32, 8, L.Q4_0) == 832
    # Registers for three waves (Q5_1, 7 heads): six workgroups per unit, not eight.
    assert plan(np.full(32, 4096), 28, 4, L.Q5_1) > plan(np.full(32, 4096), 28, 4, L.Q5_0) == 256
    # Many rounds at any size: the longest partition that leaves room for eight.
    long = plan(np.full(16, 65536), 32, 8, L.Q4_0)
    assert 640 <= long <= 1024
    assert plan(np.full(16, 65536), 64, 8, L.Q4_0) < long  # 8 heads' scores take more LDS


def test_compiled_bindings_agree_with_ctypes():
    """infer_train_amd._call passes the same arguments as the ctypes table:
    same results and statuses (nothing here reaches a device), and what ctypes
    refuses stays refused."""
    from infer_train_amd import _lib as L

    for args in ((32, 28, 128, 4097, 512), (1, 1, 128, 0, 64), (0, 1, 128, 5, 64), (65535, 64, 256, 2 ** 31 - 1, 64)):
        assert L.call.it_paged_decode_workspace(*args) == L.lib.it_paged_decode_workspace(*args)
    assert L.call.it_paged_prefill_workspace(32, 8, 1, 500, 1032, 16) == L.lib.it_paged_prefill_workspace(32, 8, 1, 500, 1032, 16) > 0
    assert L.call.it_paged_prefill_workspace(32, 8, 8, 512, 160, 16) == 0  # 512 workgroups without cuts
    assert L.call.it_paged_prefill_workspace(32, 8, 1, 4000, 250, 16) == 0  # 504 units of one sequence: no room for two cuts
    assert L.call.it_paged_prefill_workspace(16, 2, 15, 176, 127, 16) == 0 < L.call.it_paged_prefill_workspace(16, 2, 15, 176, 128, 16)
    tile = 8 * 64 * (16 * 16 + 8)  # 8 waves' partials
    assert L.call.it_paged_prefill_workspace(32, 8, 1, 64, 128, 16) == 256 + 8 * 4 * tile  # 2048 keys: 4 cuts of 8 units
    ctx, out = np.array([1024, 4096, 17], np.int32), C.c_int32()
    assert L.call.it_paged_decode_partition(L.BF16, 128, 16, 28, 4, ctx, None, 3, 256, out) == L.OK
    want = C.c_int32()
    assert L.lib.it_paged_decode_partition(L.BF16, 128, 16, 28, 4, ctx.ctypes.data, None, 3, 256, C.byref(want)) == L.OK
    assert out.value == want.value > 0
    assert L.call.it_kv_append(None, None, None, L.BF16, None, 1, None) == L.INVALID_INPUT
    assert b"NULL" in L.lib.it_last_error()
    assert L.call.it_paged_prefill_ws(None, None, L.BF16, 8, None, 1, None, 1, None, 1, 0.1, 1, None, 0, None, L.BF16,
                                      None) == L.INVALID_INPUT
    with pytest.raises(TypeError):
        L.call.it_kv_evict(None, None, 0)
    for bad in ((None, None, 1.0, None), (1.5, None, 0, None), (None, "x", 0, None)):
        with pytest.raises(C.ArgumentError):
            L.call.it_kv_evict(*bad)


def test_compiled_bindings_take_and_refuse_what_ctypes_does():
    """Arguments other than plain ints, floats and None: the compiled binding
    gives the ctypes table's result or its exception type, argument by
    argument.  No function here reaches a device: the cache is NULL, or host
    arithmetic answers."""
    import torch

    from infer_train_amd import _lib as L

    class Index:
        def __index__(self):
            return 4097

    class Parameter:
        _as_parameter_ = 4097

    def outcome(f, *args):
        try:
            return f(*args)
        except Exception as e:  # noqa: BLE001
            return type(e)

    arr = np.zeros(4, np.int32)
    odd = [np.int64(4097), np.int32(4097), np.uint8(7), torch.tensor(4097), Index(), Parameter(), C.c_int32(4097), True,
           2 ** 40 + 4097, -1, 4097.0, np.float32(3.0), None, arr, arr[:1], b"abcd", bytearray(8), [1], C.byref(C.c_int32())]
    taken = 0
    for x in odd:
        for i in range(5):
            args = [32, 28, 128, 4097, 512]
            args[i] = x
            want = outcome(L.lib.it_paged_decode_workspace, *args)
            assert outcome(L.call.it_paged_decode_workspace, *args) == want, (x, i)
            taken += not isinstance(want, type)
    assert taken >= 5 * 8  # numpy integers, a 0-d tensor, __index__, _as_parameter_, ctypes values, bool, wide and negative ints
    assert L.call.it_paged_decode_workspace(32, 28, 128, np.int64(4097), 512) == L.lib.it_paged_decode_workspace(32, 28, 128, 4097, 512)
    # Addresses (None and 0 keep the call from any device): a buffer is not one.
    for x in odd + [C.c_void_p(), C.c_void_p(64)]:
        for i in (1, 3):
            args = [None, None, 0, None]
            args[i] = x
            assert outcome(L.call.it_kv_evict, *args) == outcome(L.lib.it_kv_evict, *args), (x, i)
    for x in (arr, arr[:1], np.int64(64), bytearray(8)):
        with pytest.raises(C.ArgumentError):
            L.call.it_kv_append(None, x, None, L.BF16, None, 1, None)
    for args in ((), (32,), (32, 28, 128, 4097), (32, 28, 128, 4097, 512, 1)):
        assert outcome(L.call.it_paged_decode_workspace, *args) == outcome(L.lib.it_paged_decode_workspace, *args), args
    for scale in (1, np.float32(0.5), np.float64(0.5), torch.tensor(0.5), 10 ** 400, "0.5", None):
        args = [None, None, L.BF16, 8, None, 1, None, 1, None, 1, scale, 1, None, 0, None, L.BF16, None]
        assert outcome(L.call.it_paged_prefill_ws, *args) == outcome(L.lib.it_paged_prefill_ws, *args), scale
    # The planner's host arrays: contiguous ones are read, others are not taken.
    ctx, out = np.array([1024, 4096, 17], np.int32), C.c_int32()
    planner = [L.BF16, 128, 16, 28, 4, ctx, None, 3, 256, out]
    assert L.call.it_paged_decode_partition(*planner) == L.OK and out.value > 0
    for i, x in ((5, np.repeat(ctx, 2)[::2]), (5, np.int64(64)), (9, np.int64(64))):
        bad = list(planner)
        bad[i] = x
        with pytest.raises(C.ArgumentError):
            L.call.it_paged_decode_partition(*bad)
    for n in (np.int64(3), torch.tensor(3)):
        out.value = 0
        assert L.call.it_paged_decode_partition(*planner[:5], ctx.ctypes.data, None, n, 256, C.addressof(out)) == L.OK
        assert out.value > 0


def test_compiled_bindings_belong_to_this_interpreter(monkeypatch):
    """The binding is built with the headers of the interpreter that runs
    build(), under its ABI's name, so that another one does not load it."""
    import subprocess
    import sys
    import sysconfig

    import __graft_entry__ as entry
    from infer_train_amd import _lib as L

    assert L.call.__file__.endswith("_call" + sysconfig.get_config_var("EXT_SUFFIX"))
    calls = []
    monkeypatch.setattr(subprocess, "run", lambda cmd, **kw: calls.append(cmd))
    entry.build()
    csrc = [c for c in calls if any(x.endswith("csrc") for x in c)]
    assert len(csrc) == 1 and f"PYTHON={sys.executable}" in csrc[0]
