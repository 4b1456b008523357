"""Host-side logic (no GPU work): the package's calibration / LUT / blob
arithmetic against the reference golden vectors, the decode workspace
contract, store memory accounting on CPU tensors, and the C-ABI library
exporting every entry point include/fragpack_hip.h declares."""

from __future__ import annotations

import ctypes
from pathlib import Path
import re

import numpy as np
import pytest
import torch

from fragpack_amd.compression import attn_page as ap
from fragpack_amd.compression import attn_tables as at
from fragpack_amd.ops import fused_attn_decode as fad
from fragpack_amd.ops.fragpack_ext import LIB_PATH

ROOT = Path(__file__).resolve().parent.parent


def test_constants():
    assert ap.DENSE_BYTES == 22528 and ap.RAW_RECORD_BYTES == 32768 and ap.VAR_CAP == 2048
    assert ap.TABLE_ENTRIES == 22 and ap.BLOB_MAGIC == 0x424B5046


def test_kernel_order_and_calibration_vs_golden(golden):
    for kv in (0, 1):
        assert np.array_equal(ap.kernel_order(kv), golden[f"kernel_order_kv{kv}"])
    assert np.array_equal(ap.calibrate_table(golden["tie_input"]), golden["tie_table"])
    assert np.array_equal(at.calibrate(golden["cal_dump"]), golden["cal_table"])


def test_luts_vs_golden(golden):
    for i in range(2):
        table = golden[f"plut{i}_table"]
        assert np.array_equal(np.array(ap.primary_lut(table), np.uint32), golden[f"plut{i}"])
        assert np.array_equal(np.frombuffer(ap.secondary_lut(table), np.uint8), golden[f"slut{i}"])
    dt = at.device_tables(golden["cal_table"], torch.device("cpu"))
    assert np.array_equal(dt.rank_of.numpy(), golden["cal_rank_of"])
    assert np.array_equal(dt.plut.numpy(), golden["cal_plut"])
    assert np.array_equal(dt.slut.numpy(), golden["cal_slut"])


def test_blob_sizes_vs_golden(golden):
    for (l, h), head, slot in zip(golden["blob_geo"], golden["blob_head"], golden["blob_slot"]):
        assert ap.blob_head_bytes(int(l), int(h)) == head
        assert ap.blob_slot_bytes(int(l), int(h)) == slot


def test_tables_npz_round_trip(tmp_path):
    rng = np.random.default_rng(0)
    dump = rng.integers(0, 1 << 16, size=(2, 3, 2, 128, 4, 128), dtype=np.uint16)
    table = at.calibrate(dump)
    assert table.shape == (3, 2, 4, 22)
    path = tmp_path / "t.npz"
    np.savez(path, table=table)
    dt = at.load_tables(str(path), torch.device("cpu"), slice(2, 4))
    assert dt.rank_of.shape == (3, 2, 2, 256)
    with pytest.raises(ValueError):
        at.load_tables(str(path), torch.device("cpu"), slice(4, 8))
    with pytest.raises(ValueError):
        at.device_tables(np.zeros((1, 2, 1, 21), np.uint8), torch.device("cpu"))


def test_decode_units_and_workspace():
    assert fad.decode_units(4, 4, 256) >= 4
    assert fad.decode_units(269, 4, 256) == 269 + fad.SPLIT_WAVES * (fad.UNITS_PER_CU * 256 // 4) - 1
    opart, ml, plan = fad.workspace_elems(4, 100)
    assert opart == 4 * 100 * 8 * 128 and ml == 4 * 100 * 16
    assert plan >= 2 + 4 * 100 + 8 * 100 + 4 * 100


def test_encode_record_rejects_bad_size():
    with pytest.raises(ValueError):
        ap.encode_record(np.zeros(10, np.uint16), np.arange(22, dtype=np.uint8), 0)


def test_memory_usage_counts_page_stride_and_separates_overflow():
    """Store accounting on CPU tensors (no kernels): padded arena rows are
    counted at their stride; only the overflow pool scales with its size."""
    from fragpack_amd.ops.hbm_kv import HbmKvStore, page_bytes

    layers, blocks, heads = 2, 3, 1
    payload = page_bytes(heads)
    strides = (payload + 16, payload + 48)
    owners = [torch.empty((blocks, s), dtype=torch.uint8) for s in strides]
    arenas = [o[:, :payload] for o in owners]
    table = np.broadcast_to(np.arange(22, dtype=np.uint8), (layers, 2, heads, 22)).copy()
    tables = at.device_tables(table, torch.device("cpu"))

    def build(n):
        return HbmKvStore(arenas, heads, tables, max_tokens=128, staging_slots=2, overflow_records=n)

    small, larger = build(1).memory_usage(), build(2).memory_usage()
    assert small["arena"] == sum(o.numel() for o in owners) > layers * blocks * payload
    assert small["staging"] > 0 and small["scratch"] > 0 and small["metadata"] > 0 and small["codebooks"] > 0
    assert larger["overflow"] == 2 * small["overflow"]
    assert {k: v for k, v in small.items() if k != "overflow"} == {k: v for k, v in larger.items() if k != "overflow"}


def test_store_rejects_mismatched_tables():
    from fragpack_amd.ops.hbm_kv import HbmKvStore

    tables = at.device_tables(np.zeros((1, 2, 2, 22), np.uint8) + np.arange(22, dtype=np.uint8), torch.device("cpu"))
    with pytest.raises(ValueError):
        HbmKvStore([torch.empty((2, 64), dtype=torch.uint8)] * 2, 2, tables, 128, 1, 1)


def _declared_symbols():
    text = (ROOT / "include" / "fragpack_hip.h").read_text()
    return sorted(set(re.findall(r"^\s*(?:int|int64_t|const char\*)\s+(fp_\w+)\s*\(", text, re.M)))


def test_library_exports_every_declared_symbol():
    assert LIB_PATH.exists(), "build the library first (__graft_entry__.build())"
    lib = ctypes.CDLL(str(LIB_PATH))
    syms = _declared_symbols()
    assert len(syms) >= 12
    for name in syms:
        assert hasattr(lib, name), name
    lib.fp_abi_version.restype = ctypes.c_int
    assert lib.fp_abi_version() == 1
    lib.fp_last_error.restype = ctypes.c_char_p
    assert isinstance(lib.fp_last_error(), bytes)


def test_c_abi_rejects_bad_arguments_without_gpu_work():
    """Argument checks run before any launch: errors come back as -1 + message."""
    lib = ctypes.CDLL(str(LIB_PATH))
    lib.fp_last_error.restype = ctypes.c_char_p
    f = lib.fp_fused_decode
    f.restype = ctypes.c_int
    p, i64 = ctypes.c_void_p, ctypes.c_int64
    f.argtypes = [p, i64, i64, i64, i64, p, p, p, p, p, i64, p, p, i64, p, i64, p, i64, p, i64, i64, ctypes.c_int,
                  ctypes.c_double, p]
    # group 3 does not divide 8
    rc = f(None, 1024, 1, 4, 3, None, None, None, None, None, 1, None, None, 0, None, 0, None, 0, None, 1024, 1, 1,
           0.1, None)
    assert rc == -1 and b"group" in lib.fp_last_error()
    # units < batch
    rc = f(None, 4096, 4, 4, 8, None, None, None, None, None, 1, None, None, 1 << 20, None, 1 << 20, None, 1 << 20,
           None, 4096, 2, 1, 0.1, None)
    assert rc == -1 and b"unit" in lib.fp_last_error()
    # empty batch is a no-op
    assert f(None, 4096, 0, 4, 8, None, None, None, None, None, 1, None, None, 0, None, 0, None, 0, None, 4096, 0, 1,
             0.1, None) == 0


def test_store_write_rejects_bad_steps_without_gpu_work():
    """The store write's argument checks (fp_store.hip write_args) return -1
    with a message before any launch: a step of 2^30+ (token, head) items,
    odd strides; an empty step is a no-op."""
    from fragpack_amd.ops.fragpack_ext import FpStore

    lib = ctypes.CDLL(str(LIB_PATH))
    lib.fp_last_error.restype = ctypes.c_char_p
    f = lib.fp_hbm_write
    f.restype = ctypes.c_int
    p, i64 = ctypes.c_void_p, ctypes.c_int64
    f.argtypes = [ctypes.POINTER(FpStore), p, i64, i64, p, i64, i64, p, i64, i64, p]
    d = FpStore(num_layers=1, num_blocks=4, kv_heads=8, staging_slots=2, scratch_slots=2, ovf_words=1, list_cap=64,
                overflow_records=32)
    dummy = p(256)  # never dereferenced: the checks fail first
    rc = f(ctypes.byref(d), dummy, 8 * 128, 128, dummy, 8 * 128, 128, dummy, 1 << 27, 0, None)
    assert rc == -1 and b"items" in lib.fp_last_error()
    rc = f(ctypes.byref(d), dummy, 8 * 128 + 1, 128, dummy, 8 * 128, 128, dummy, 16, 0, None)
    assert rc == -1 and b"strides" in lib.fp_last_error()
    rc = f(ctypes.byref(d), dummy, 8 * 128, 128, dummy, 8 * 128, 128, dummy, 16, 5, None)
    assert rc == -1 and b"layer" in lib.fp_last_error()
    assert f(ctypes.byref(d), dummy, 8 * 128, 128, dummy, 8 * 128, 128, dummy, 0, 0, None) == 0


def test_planner_reciprocal_division_is_exact_within_its_range():
    """The device planners divide x / d (0 <= x < 2^22, d >= 1) by a float
    product with the hardware reciprocal (relative error up to one ulp,
    2^-23) and one correction step each way (fp_attn.hip, ``Divider``).
    Restated in float32 with the reciprocal taken one ulp low, exact and one
    ulp high: the quotient equals x // d everywhere sampled, including
    multiples of d and their neighbours and the range's ends."""
    rng = np.random.default_rng(7)
    ds = np.concatenate([np.arange(1, 3000), rng.integers(3000, 1 << 22, 4000), [(1 << 22) - 1]]).astype(np.int64)
    for d in ds:
        k = rng.integers(0, ((1 << 22) - 1) // d + 1, 24)
        x = np.concatenate([k * d, k * d - 1, k * d + d - 1, rng.integers(0, 1 << 22, 24), [0, (1 << 22) - 1]])
        x = x[(x >= 0) & (x < (1 << 22))]
        exact = np.float32(1.0) / np.float32(d)
        for inv in (np.nextafter(exact, np.float32(0)), exact, np.nextafter(exact, np.float32(2))):
            q = np.trunc(x.astype(np.float32) * np.float32(inv)).astype(np.int64)
            q += (q + 1) * d <= x
            q -= q * d > x
            np.testing.assert_array_equal(q, x // d, err_msg=f"d={d}")


def test_plan_reuse_without_a_plan_is_refused():
    """A reusing decode call (replan=False) on a workspace no planning call
    has written is refused on the host, before any device pointer is taken:
    the kernel would follow whatever descriptors the buffer holds."""
    from fragpack_amd.ops.fragpack_ext import extension

    B, H, G, units = 2, 2, 8, 8
    q = torch.zeros((B, H * G, 128), dtype=torch.bfloat16)
    out = torch.zeros_like(q)
    opart, ml, plan = fad.workspace_elems(H, units)
    ws = (torch.zeros(opart), torch.zeros(ml), torch.zeros(plan, dtype=torch.int32))
    args = (q, torch.zeros((4, 2, H), dtype=torch.int64), torch.zeros((4, 2, H), dtype=torch.int32),
            torch.zeros((2, H, 2), dtype=torch.int32), torch.zeros((2, H, 16), dtype=torch.uint8),
            torch.zeros((B, 4), dtype=torch.int32), torch.ones(B, dtype=torch.int32), *ws, out, units)
    with pytest.raises(RuntimeError, match="plan first"):
        extension().fused_decode(*args, False, 0.1, G)
    # a key from another shape is refused too
    ws[2]._fp_plan_key = (units + 1, B, H)
    with pytest.raises(RuntimeError, match="plan first"):
        extension().fused_decode(*args, False, 0.1, G)


def prefill_plan(heads, group, seqs, total_q, max_q, max_k, causal=True, cus=256):
    """(waves, split workgroups, workgroups of a row, rows, tile-major) of a prefill call on ``cus`` compute units."""
    lib = ctypes.CDLL(str(LIB_PATH))
    lib.fp_prefill_plan.argtypes = [ctypes.c_int64] * 6 + [ctypes.c_int, ctypes.c_int64, ctypes.c_void_p]
    plan = (ctypes.c_int64 * 5)()
    assert lib.fp_prefill_plan(heads, group, seqs, total_q, max_q, max_k, int(causal), cus, plan) == 0
    return tuple(plan)


@pytest.mark.parametrize("heads", [1, 2, 4, 5, 6, 8, 12, 16, 64])
@pytest.mark.parametrize("seqs,tiles", [(1, 1), (3, 11), (4, 1 << 18), (512, 2048), (8, (1 << 20) - 1), (1, (1 << 23) - 1)])
def test_prefill_grid_covers_the_tiles_within_the_launch_limit(heads, seqs, tiles):
    """HIP takes fewer than 2^32 work items along x: one head's tiles fit up to
    2^23 - 1 workgroups of 512, so that many are never refused, and the rows
    hold every (query tile, head)."""
    waves, _, row, rows, _ = prefill_plan(heads, 8, seqs, 0, 32 * tiles, 4096)
    assert row * 64 * waves < 1 << 32
    assert rows <= heads and heads % rows == 0
    per_head = seqs * tiles * (8 // waves)
    assert per_head * (heads // rows) <= row < per_head * (heads // rows) + 8 * (heads // rows)


def test_no_call_below_the_split_key_bound_splits():
    """The bound below which a caller need not ask for a workspace is the
    launch rule's own: nothing below it splits, one row a key tile past it does."""
    from fragpack_amd.ops.fragpack_ext import extension

    ext = extension()
    least = ext._lib.fp_prefill_split_min_keys()
    assert ext._split_keys == least and prefill_plan(1, 8, 1, 1, 1, least + 64)[1] == 256
    rng = np.random.default_rng(5)
    for _ in range(2000):
        heads, group, seqs = int(rng.integers(1, 33)), int(2 ** rng.integers(0, 4)), int(rng.integers(1, 9))
        max_q = int(np.exp(rng.uniform(0, 9)))
        total = int(rng.integers(max_q, seqs * max_q + 1))
        assert prefill_plan(heads, group, seqs, total, max_q, int(rng.integers(1, least)))[1] == 0
        assert prefill_plan(heads, group, seqs, 0, max_q, 1 << 20)[1] == 0  # no rows given: never split


def test_one_workspace_serves_every_split_call():
    """The largest workspace of any call of up to max_k keys holds what each
    such call asks for: the sizes here are the library's for 256 CUs, whose
    part slots and key-tile entries are 2 x 133120 + 32 and 1032 bytes."""
    lib = ctypes.CDLL(str(LIB_PATH))
    i64 = ctypes.c_int64
    lib.fp_prefill_workspace_most.argtypes, lib.fp_prefill_workspace_most.restype = [i64, i64], i64
    lib.fp_prefill_split_min_keys.restype = i64
    assert lib.fp_prefill_workspace_most(lib.fp_prefill_split_min_keys() - 1, 256) == 0
    rng = np.random.default_rng(6)
    for _ in range(2000):
        heads, group, seqs = int(rng.integers(1, 33)), int(2 ** rng.integers(0, 4)), int(rng.integers(1, 5))
        max_q, max_k = int(np.exp(rng.uniform(0, 8))), int(np.exp(rng.uniform(7.5, 13)))
        total = int(rng.integers(max_q, seqs * max_q + 1))
        if prefill_plan(heads, group, seqs, total, max_q, max_k)[1]:
            rows = 256 // group
            tiles = min(seqs * -(-max_q // rows), total // rows + seqs) * heads
            need = 256 * (2 * 133120 + 32) + tiles * -(-max_k // 64) * 1032
            assert need <= lib.fp_prefill_workspace_most(max_k, 256)


@pytest.mark.parametrize("heads,group,q_lens,k_lens,causal,waves", [
    (16, 1, [2048, 2048], [2048, 2048], True, 4),  # fresh prompts: tiles of unequal length
    (16, 1, [2048, 2048], [2048, 2048], False, 8),  # full attention: all equal, 256 of them
    (5, 4, [2048] * 2, [2048] * 2, False, 4),  # 320: more than a round
    (8, 4, [1024], [1024], False, 4),  # few tiles: 8 waves would leave CUs idle
    (20, 1, [128] * 8, [1128] * 8, True, 8),  # 160 tiles, one a sequence, several rows of heads
    (5, 4, [64] * 32, [564] * 32, True, 8),
    (5, 4, [64] * 24, [564] * 24, True, 4),  # 120: CUs would idle
    (8, 4, [64] * 20, [564] * 20, True, 4),  # 160, one row
    (10, 4, [128] * 8, [1128] * 8, True, 8),  # 160, two a sequence
    (20, 1, [1024] * 2, [4096] * 2, True, 4),  # 160, four a sequence
])
def test_prefill_waves(heads, group, q_lens, k_lens, causal, waves):
    assert prefill_plan(heads, group, len(q_lens), sum(q_lens), max(q_lens), max(k_lens), causal)[0] == waves


@pytest.mark.parametrize("heads,q_lens,k_lens,turns", [
    (5, [2048] * 4, [2048] * 4, True),
    (5, [2048, 2048, 2048, 2000], [2048] * 4, False),  # lengths differ
    (5, [2048], [2048], False),
    (8, [2048] * 4, [2048] * 4, False),  # a head per XCD
    (3, [1024] * 4, [9216] * 4, False),  # one round
    (3, [4096] * 4, [12288] * 4, True),
    (4, [512] * 4, [512] * 4, False),  # a workgroup per CU
])
def test_prefill_sequences_take_turns(heads, q_lens, k_lens, turns):
    assert prefill_plan(heads, 4, len(q_lens), sum(q_lens), max(q_lens), max(k_lens))[4] == turns
