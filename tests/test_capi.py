"""The C ABI library (CPU-side checks: loads, exports every declared symbol,
validates arguments before touching a device)."""
import ctypes
import re
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


def declared_symbols():
    text = (ROOT / "include" / "cda_hip.h").read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(cda_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    from sub0_amd import _native
    L = _native.lib()
    syms = declared_symbols()
    assert len(syms) >= 7
    for s in syms:
        assert hasattr(L, s), s
    assert sorted(_native.SYMBOLS) == syms


def test_version_and_plan():
    from sub0_amd import _native
    assert _native.lib().cda_hip_version() >= 100
    tile, splits = _native.decode_plan(32, 32, 8, 65536)
    assert tile % 32 == 0 and tile * splits >= 65536 and splits <= 512
    tile, splits = _native.decode_plan(1, 32, 8, 4096, 100)
    assert tile == 128 and splits == 32
    assert _native.decode_plan(1, 32, 8, 0) == (32, 1)
    ws1 = _native.decode_workspace_size(4, 32, 8, 4096)
    ws2 = _native.decode_workspace_size(4, 32, 8, 65536)
    assert 0 < ws1 <= ws2 and ws1 % 256 == 0


def test_decode_fused_plan_fits_the_workspace():
    """The single-launch plan (256 CUs without a device): whole 64-token
    chunks per wave, at most 4096 pages per workgroup, every token covered,
    and never more splits than the three-launch plan, whose
    cda_decode_workspace_size() callers allocate."""
    from sub0_amd import _native
    assert _native.decode_fused_plan(32, 8, 65536) == (8192, 1)     # one launch per step
    assert _native.decode_fused_plan(32, 8, 4096) == (512, 1)
    assert _native.decode_fused_plan(1, 8, 4096) == (64, 8)         # one chunk per wave
    assert _native.decode_fused_plan(1, 8, 65536) == (256, 32)
    assert _native.decode_fused_plan(4, 8, 65536) == (1024, 8)
    assert _native.decode_fused_plan(32, 8, 262144) == (8192, 4)    # page-row table cap
    assert _native.decode_fused_plan(3, 8, 0) == (64, 1)
    for B in (1, 2, 3, 4, 5, 7, 8, 16, 31, 32, 64, 256):
        for n in (1, 63, 64, 65, 511, 512, 513, 1000, 4096, 16383, 16384, 65535, 65536,
                  65537, 131072, 262144, 1000003):
            wt, ns = _native.decode_fused_plan(B, 8, n)
            assert wt % 64 == 0 and 64 <= 8 * wt <= 65536, (B, n, wt)
            assert 8 * wt * ns >= n and 8 * wt * (ns - 1) < n, (B, n, wt, ns)
            _, ns3 = _native.decode_plan(B, 8 * 4, 8, n)
            assert ns <= ns3, (B, n, ns, ns3)
    with pytest.raises(ValueError):
        _native.decode_fused_plan(0, 8, 100)


def test_decode_fused_plan_is_the_cheapest_and_quick():
    """The plan's search over round boundaries finds what trying every number of
    chunks per wave finds (256 CUs; least rounds x (k + 3), in half chunks, 3 for
    a combine; the largest k of equals), and a long context's plan, made on every
    call, costs the host no more than a short one's (trying all 128 took 0.8 us
    at 64K tokens; the least of 40 batches is compared, with 0.4 us allowed)."""
    import time
    from sub0_amd import _native

    def every_k(B, H, n):
        chunks, units, limit = max(1, -(-n // 512)), B * H, _native.decode_plan(B, H, H, n)[1]
        best = None
        for k in range(min(128, chunks), 0, -1):
            ns = -(-chunks // k)
            if ns > limit and best is not None:
                break
            cost = 2 * -(-units * ns // 256) * (k + 3) + (3 if ns > 1 else 0)
            if best is None or cost < best[0]:
                best = (cost, 64 * k, ns)
        return best[1:]

    for B in (1, 2, 3, 5, 8, 12, 16, 31, 33, 64, 65, 257):
        for H in (1, 2, 3, 8, 16):
            for n in (0, 1, 512, 513, 1500, 4096, 7000, 16384, 30001, 65536, 100000, 131073,
                      1000003, 40000000):
                assert _native.decode_fused_plan(B, H, n) == every_k(B, H, n), (B, H, n)

    L = _native.lib()
    out = [ctypes.byref(ctypes.c_int32()) for _ in range(2)]

    def host_time(n):
        best = float("inf")
        for _ in range(40):
            t = time.perf_counter()
            for _ in range(500):
                L.cda_decode_fused_plan(1, 8, n, *out)
            best = min(best, time.perf_counter() - t)
        return best / 500
    assert host_time(65536) - host_time(512) < 0.4e-6


def test_decode_deal_by_length_fits_the_merge():
    """Where slots are dealt by length, the deal the kernel makes (the smallest
    k whose splits of 512 * k tokens fit the B * n_splits slots, if below the
    even split's) fits them for one long sequence among short ones, and gives
    no sequence more than the 1024 splits that the merge holds."""
    from sub0_amd import _native
    dealt = 0
    lengths = sorted({(1 << e) + d for e in range(11, 25) for d in (0, 1, 1 << (e - 1))}
                     | {1440000, 2030000})
    for H in (1, 2, 4, 8, 16):
        for B in (8, 9, 12, 16, 23, 32, 48, 63, 64):
            for n in lengths:
                if not _native.decode_deals_by_length(B, H, n):
                    continue
                dealt += 1
                wave_tokens, ns = _native.decode_fused_plan(B, H, n)
                for long in {n, n // 2 + 1025, n // 3, min(n, 512 * (B * ns - B + 1))}:
                    chunks = [-(-long // 512)] + [1] * (B - 1)
                    k = next((k for k in range(1, 129)
                              if sum(max(1, -(-c // k)) for c in chunks) <= B * ns),
                             wave_tokens // 64)
                    k = min(k, wave_tokens // 64)
                    counts = [max(1, -(-c // k)) for c in chunks]
                    assert sum(counts) <= B * ns, (H, B, n, long, k)
                    assert max(counts) <= 1024, (H, B, n, long, k, max(counts))
    assert dealt > 100
    # Both sides of the measured line.
    for B, H, n, plan, on in ((16, 2, 16384, (4, 8), True), (12, 4, 8192, (4, 4), False),
                              (32, 1, 16384, (4, 8), False), (48, 1, 12288, (5, 5), False),
                              (12, 4, 12288, (5, 5), False), (12, 1, 60000, (6, 20), True),
                              (64, 1, 12288, (6, 4), False), (12, 8, 8192, (8, 2), False),
                              (9, 8, 12288, (8, 3), True), (64, 1, 16384, (8, 4), True),
                              (12, 8, 16384, (16, 2), True), (8, 2, 16384, (2, 16), False)):
        wave_tokens, ns = _native.decode_fused_plan(B, H, n)
        assert (wave_tokens // 64, ns) == plan, (B, H, n)           # chunks per wave, splits
        assert _native.decode_deals_by_length(B, H, n) is on, (B, H, n)
    assert not _native.decode_deals_by_length(65, 1, 65536)     # a lane per sequence
    with pytest.raises(ValueError):
        _native.decode_deals_by_length(0, 8, 100)


def test_prefill_key_split_plan():
    """Host-side plan of the key-split prefill: split only short chunks over
    long contexts (grid under 256 workgroups, >= 4 key tiles per split, <= 64
    splits); the workspace holds (O, m, l) per split, query row and q-head."""
    from sub0_amd import _native
    ws = _native.prefill_workspace_size
    # 16 queries over 16K keys, 8 KV heads: 8 workgroups -> 32 splits of 8 tiles.
    assert ws(1, 16, 32, 8, 16, 16384) == 32 * 16 * 32 * 128 * 4 + 32 * 16 * 32 * 2 * 4
    # 1 query over 64K keys, 1 KV head: 1 workgroup -> min(256, 1024 // 4) -> 64 (the cap).
    assert ws(1, 1, 4, 1, 1, 65536) == 64 * 1 * 4 * 128 * 4 + 64 * 1 * 4 * 2 * 4
    # 4000 keys = 63 tiles: min(64, 63 // 4) = 15 splits -> 5 tiles each -> 13 splits.
    assert ws(1, 16, 32, 8, 16, 4000) == 13 * 16 * 32 * 128 * 4 + 13 * 16 * 32 * 2 * 4
    assert ws(1, 16, 32, 8, 16, 200) == 0            # too few keys to split
    # 300 queries x 2 over 5000 keys: 80 workgroups of 79 tiles -> 3 splits of
    # 27 (one round of 240), not 4 of 20 (320 workgroups, two rounds).
    assert ws(2, 600, 32, 8, 300, 5000) == 3 * 600 * 32 * 128 * 4 + 3 * 600 * 32 * 2 * 4
    # 100 queries x 3 over 4100 keys: 48 workgroups of 65 tiles -> 5 splits of 13.
    assert ws(3, 300, 32, 8, 100, 4100) == 5 * 300 * 32 * 128 * 4 + 5 * 300 * 32 * 2 * 4
    # The partials' traffic counts: 64 queries x 12 over 16K keys, 96 workgroups
    # of 257 tiles -> 5 splits of 52 (two rounds), not 8 of 33 (three); x 28, 224
    # workgroups -> unsplit, not 8 splits.
    assert ws(12, 768, 32, 8, 64, 16448) == 5 * 768 * 32 * 128 * 4 + 5 * 768 * 32 * 2 * 4
    assert ws(28, 1792, 32, 8, 64, 16448) == 0
    # Fewer rows than the bound: 389, 245, 215 queries over 4.4K keys, 144
    # workgroups by the bound but about 15 blocks x 8 heads: 2 splits fit one round,
    # where equal counts (21 blocks) take 3 of 23 tiles in two.
    assert ws(3, 849, 32, 8, 389, 4400) == 2 * 849 * 32 * 128 * 4 + 2 * 849 * 32 * 2 * 4
    assert ws(3, 1167, 32, 8, 389, 4400) == 3 * 1167 * 32 * 128 * 4 + 3 * 1167 * 32 * 2 * 4
    assert ws(8, 8 * 4096, 32, 8, 4096, 8192) == 0   # config-3-sized grid fills the chip
    assert ws(0, 0, 32, 8, 16, 16384) == 0
    assert ws(1, 16, 32, 5, 16, 16384) == 0          # group size not 4 or 8


def test_invalid_arguments_are_rejected_before_launch():
    from sub0_amd import _native
    L = _native.lib()
    P = ctypes.c_void_p
    dummy = P(256)
    rc = L.cda_decode_full_hmma_v3(dummy, dummy, 16, 144, 8, dummy, 1, dummy, dummy, dummy, 16,
                                   dummy, None, dummy, 1, 32, 3, 16, 0, 16, 0.1, dummy, 1 << 20,
                                   None)
    assert rc == -1 and b"group_size" in L.cda_hip_last_error()
    rc = L.cda_decode_full_hmma_v3(dummy, dummy, 16, 144, 8, dummy, 1, dummy, dummy, dummy, 16,
                                   dummy, None, dummy, 1, 32, 4, 8, 0, 16, 0.1, dummy, 1 << 20,
                                   None)
    assert rc == -1 and b"block_size" in L.cda_hip_last_error()
    rc = L.cda_decode_full_hmma_v3(dummy, dummy, 16, 144, 8, dummy, 1, dummy, dummy, dummy, 16,
                                   dummy, None, dummy, 1, 32, 4, 16, 0, 16, 0.1, P(512), 16, None)
    assert rc == -3
    rc = L.cda_paged_encode_fused(dummy, dummy, 1024, 1024, dummy, 4, dummy, 16, 144, 8, dummy,
                                  dummy, 5, None)
    assert rc == -1 and b"levels" in L.cda_hip_last_error()
    rc = L.cda_paged_encode_fused(dummy, dummy, 1024, 1024, dummy, 4, dummy, 16, 72, 8, dummy,
                                  dummy, 16, None)
    assert rc == -1 and b"slot_bytes" in L.cda_hip_last_error()
    assert L.cda_paged_encode_fused(None, None, 0, 0, None, 0, None, 0, 0, 0, None, None, 16,
                                    None) == 0          # zero tokens: nothing to do
    assert L.cda_decode_set_timing_events(dummy, None) == -1


def test_prefill_arguments_are_rejected_before_launch():
    from sub0_amd import _native
    L = _native.lib()
    P = ctypes.c_void_p
    d = P(256)

    def call(slot_bytes, block_size, cache=d):
        return L.cda_prefill_paged_hadamard(d, cache, 64, slot_bytes, 8, d, 4, d, d, 1, d, d, 16,
                                            d, 8, 32, block_size, 8, 0.1, None)
    assert call(144, 24) == -1 and b"multiple of 16" in L.cda_hip_last_error()
    assert call(128, 16) == -1 and b"slot" in L.cda_hip_last_error()
    assert call(144, 16, P(260)) == -1 and b"aligned" in L.cda_hip_last_error()


def test_prefill_dense_checks_without_queries():
    """max_query_len 0 does not skip the checks of the loader and the attention
    that the two-call bridge made (a slot too small for the layout)."""
    from sub0_amd import _native
    L = _native.lib()
    d = ctypes.c_void_p(256)

    def call(slot_bytes, max_query_len):
        return L.cda_prefill_dense_hadamard(d, d, 64, slot_bytes, 8, d, 4, d, d, 1, d, d, 16, d, 8,
                                            32, 16, max_query_len, 64, 0.1, d, 1 << 30, None)
    for max_query_len in (8, 0):
        assert call(128, max_query_len) == -1 and b"slot" in L.cda_hip_last_error()


def test_python_binding_refuses_cpu_tensors():
    import torch
    from sub0_amd import _native
    x = torch.zeros(4, 8, 128, dtype=torch.float16)
    with pytest.raises(ValueError, match="GPU"):
        _native.paged_encode(x, x, torch.zeros(4, dtype=torch.int32),
                             torch.zeros(4, 8, 144, dtype=torch.uint8),
                             torch.zeros(16), torch.zeros(16))


def test_decode_wrapper_passes_the_table_width(monkeypatch):
    """A column slice of a block table is handed over with its stride and its
    width: the single launch reads entries before it knows the lengths, and the
    slice's last row may end where its memory does."""
    import torch
    from sub0_amd import _native
    calls = {}

    class Recorder:
        def __getattr__(self, name):
            return lambda *args: calls.__setitem__(name, args) or 0

    monkeypatch.setattr(_native, "lib", Recorder)
    monkeypatch.setattr(_native, "_require_gpu", lambda *ts: ts[0].device)
    monkeypatch.setattr(_native, "_stream", lambda dev: None)
    q = torch.zeros(3, 32, 128, dtype=torch.float16)
    cb = torch.zeros(16)
    table = torch.zeros(3, 20, dtype=torch.int32)[:, 15:]
    _native.decode(q, torch.zeros(16, 8, 144, dtype=torch.uint8), table,
                   torch.zeros(3, dtype=torch.int32), cb, cb, torch.zeros(128, 128), None,
                   torch.zeros_like(q), group_size=4, block_size=16, tile_n=0, max_seq_len=80,
                   scale=1.0)
    assert calls["cda_decode_full_hmma_v3_table"][6:8] == (20, 5)
