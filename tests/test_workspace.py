"""The workspace cache of vmk.api on the CPU: allocation, capture state and the device drain are stubbed, so the
rules themselves are checked without a GPU: geometric growth, outgrown buffers freed unless a graph was captured
over them, growth refused during capture, and a failed call setting its buffer aside only after a launch error."""
import os

import pytest
import torch

from vmk import api, lib


@pytest.fixture
def cache(monkeypatch):
    state = dict(capturing=False, drains=0)
    monkeypatch.setattr(api, "_ws", {})
    monkeypatch.setattr(api, "_captured", set())
    monkeypatch.setattr(api, "_retired", [])
    monkeypatch.setattr(api, "_alloc", lambda n, key: torch.zeros(n, dtype=torch.uint8))
    monkeypatch.setattr(api, "_capturing", lambda: state["capturing"])

    def drain(key):
        state["drains"] += 1
    monkeypatch.setattr(api, "_drain", drain)
    monkeypatch.setattr(api, "_dev_index", lambda device: 0)
    return state


def test_growth_is_geometric_and_outgrown_buffers_are_freed(cache):
    a = api.workspace(100, "cuda:0")
    assert a.numel() == api.MIN_WORKSPACE
    assert api.workspace(api.MIN_WORKSPACE, "cuda:0") is a              # fits: same buffer
    sizes = []
    need = api.MIN_WORKSPACE
    for _ in range(40):                                                   # a cache that grows a little per call
        need += api.MIN_WORKSPACE // 4
        sizes.append(api.workspace(need, "cuda:0").numel())
    grown = sorted(set(sizes))
    assert all(b >= 2 * a for a, b in zip(grown, grown[1:]))              # each growth at least doubles
    assert len(grown) <= 4
    assert api._retired == []                                             # nothing captured: nothing retained
    assert cache["drains"] == len(grown)                                  # each outgrown buffer after a drain


def test_buffer_of_a_captured_graph_is_kept(cache):
    a = api.workspace(1 << 20, "cuda:0")
    cache["capturing"] = True
    assert api.workspace(1 << 19, "cuda:0") is a                          # a capture uses the current buffer
    with pytest.raises(lib.VmkError, match="during HIP graph capture"):
        api.workspace(4 << 20, "cuda:0")                                  # growth refused while capturing
    cache["capturing"] = False
    b = api.workspace(4 << 20, "cuda:0")
    assert b is not a and api._retired == [a]                             # the graph's buffer stays alive
    c = api.workspace(16 << 20, "cuda:0")
    assert c is not b and api._retired == [a]                             # b was never captured: freed


def test_failed_call_sets_aside_only_after_a_launch_error(cache, monkeypatch):
    class Dev:
        index = 0

    class Buf:
        device = Dev()
    buf = Buf()
    api._ws[0] = buf

    def fail(code):
        def call(name, *args):
            raise lib.VmkError("boom", code=code)
        return call
    monkeypatch.setattr(lib, "call", fail(lib.REJECTED))
    with pytest.raises(lib.VmkError):
        api._launch("vmk_x", buf)
    assert api._ws[0] is buf                                              # refused on the host: kept in use
    monkeypatch.setattr(lib, "call", fail(lib.LAUNCH_ERROR))
    with pytest.raises(lib.VmkError):
        api._launch("vmk_x", buf)
    assert 0 not in api._ws and api._retired == []                        # set aside and released after a drain
    assert cache["drains"] == 1
    assert api.workspace(1 << 20, "cuda:0") is not buf                    # the next call starts from a fresh one


def test_error_codes_are_kept():
    e = lib.VmkError("x", code=2)
    assert e.code == lib.LAUNCH_ERROR and isinstance(e, RuntimeError)
    assert lib.VmkError("y").code is None


@pytest.mark.parametrize("op,heads", [("decode", (32, 8)), ("decode", (16, 1)), ("decode", (96, 4)),
                                      ("decode", (64, 1)), ("paged", (32, 8)), ("paged", (8, 1)), (2, (32, 8)),
                                      (7, (32, 8)), (8, (32, 8)), (9, (32, 8)), (16, (32, 8)), (16, (4, 1)),
                                      (64, (32, 8))])
def test_sizes_grow_with_the_batch_and_the_cache(op, heads):
    """A workspace sized for the largest batch and cache serves every smaller call: the sizes never fall as either
    grows.  Sizes around tiles, splits and the lengths at which the split size steps up."""
    if not os.path.exists(lib.LIB_PATH):
        pytest.skip("libvmk.so not built")
    so = lib.load()

    def size(B, L):
        if op == "decode":
            return so.vmk_decode_workspace_size(B, *heads, 128, L)
        if op == "paged":
            return so.vmk_decode_paged_workspace_size(B, *heads, 128, 32, -(-L // 32))
        return so.vmk_spec_workspace_size(B, op, *heads, 128, L)
    batches = [1, 2, 3, 4, 5, 7, 8, 9, 15, 16, 17, 31, 32, 33, 64, 65, 128, 300]
    lengths = sorted({max(64, base + d) for base in (64, 100, 1024, 2048, 4096, 8192, 16384, 20480, 32768, 40960, 65536,
                                                     131072, 262144, 1 << 20) for d in (-1, 0, 1, 33)})
    table = [[size(B, n) for n in lengths] for B in batches]
    assert all(v > 0 for row in table for v in row)
    for i, row in enumerate(table):
        for j in range(1, len(row)):
            assert row[j] >= row[j - 1], (batches[i], lengths[j - 1], lengths[j])
        if i:
            assert all(a >= b for a, b in zip(row, table[i - 1])), (batches[i - 1], batches[i])
