"""The allocation-free spec entry point (vmk_spec_verify_noalloc, C-ABI through ctypes) against vmk_spec_verify on
the same inputs: the same kernels and plan, so the outputs must be bit-equal.  Two calls in a row, the second on a
smaller shape (the static scratch keeps the first call's partials), and then a third at the C4 size."""
import pytest
import torch

from vmk import lib
from vmk.ops import spec

pytestmark = pytest.mark.gpu


def call_noalloc(inp, out):
    q, k, v = inp["q"], inp["k"], inp["v"]
    words = spec.mask_words(inp["bits"], q.shape[1]).contiguous()
    B, kd, Hq, D = q.shape
    lib.call("vmk_spec_verify_noalloc", q.data_ptr(), k.data_ptr(), v.data_ptr(), words.data_ptr(), out.data_ptr(),
             B, kd, Hq, k.shape[1], D, k.shape[2], words.shape[2], torch.cuda.current_stream().cuda_stream)


def call_workspace(inp):
    import vmk
    q = inp["q"]
    return vmk.spec_verify(q, inp["k"], inp["v"], spec.mask_words(inp["bits"], q.shape[1]).contiguous())


@pytest.mark.parametrize("shapes", [[(dict(B=4, L=32768, k=8), "chain", 1), (dict(B=2, L=3000, k=5), "randn", 2),
                                     (dict(B=2, L=65536, k=64), "tree_bd", 3)]])
def test_noalloc_equals_workspace_entry_point(shapes):
    for shape, dist, seed in shapes:
        print(f"noalloc spec {shape} {dist} seed={seed}", flush=True)
        inp = spec.make_inputs(shape, seed=seed, dist=dist, device="cuda")
        out = torch.full_like(inp["q"], float("nan"))
        call_noalloc(inp, out)
        want = call_workspace(inp)
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), want.view(torch.int16)), shape


def test_noalloc_refuses_shapes_beyond_its_scratch():
    """A shape whose partials exceed the scratch is refused before anything is launched (the tensors are tiny: the
    call must not read them)."""
    x = torch.zeros(16, dtype=torch.float16, device="cuda")
    words = torch.zeros(16, dtype=torch.int32, device="cuda")
    L = 64 * 2 ** 20                                   # 16 splits x 256 items x 128 KiB of partials per 4096 keys
    with pytest.raises(lib.VmkError, match="static scratch"):
        lib.call("vmk_spec_verify_noalloc", x.data_ptr(), x.data_ptr(), x.data_ptr(), words.data_ptr(), x.data_ptr(),
                 8, 64, 32, 8, 128, L, 2, torch.cuda.current_stream().cuda_stream)


def test_noalloc_on_a_side_stream():
    """The scratch is looked up for the device of the stream the call is launched on (here a non-default stream
    of the current GPU), through the Python wrapper, and gives the same bits as the workspace entry point."""
    import vmk
    inp = spec.make_inputs(dict(B=2, L=5000, k=8), seed=4, dist="chain", device="cuda")
    words = spec.mask_words(inp["bits"], 8).contiguous()
    want = call_workspace(inp)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        out = torch.full_like(inp["q"], float("nan"))
        vmk.spec_verify_noalloc(inp["q"], inp["k"], inp["v"], words, out)
    torch.cuda.synchronize()
    assert torch.equal(out.view(torch.int16), want.view(torch.int16))


def launches(call):
    """Launches of one call, as nodes of its HIP graph."""
    import ctypes
    import glob
    import os
    path = glob.glob(os.path.join(os.path.dirname(torch.__file__), "lib", "libamdhip64.so*"))[0]   # the one in use
    hip = ctypes.CDLL(path)
    call()                                             # what is looked up once is looked up before the capture
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        call()
    n = ctypes.c_size_t()
    assert hip.hipGraphGetNodes(ctypes.c_void_p(graph.raw_cuda_graph()), None, ctypes.byref(n)) == 0
    return n.value


@pytest.mark.parametrize("shape,want_launches", [
    (dict(B=2, L=8192, k=16), 2),         # as units its partials would not fit: splits, not steps of units
    (dict(B=4, L=3000, k=9, Hkv=4, Hq=16), 2),
    (dict(B=1, L=8192, k=16), 2),         # units that fit
    (dict(B=32, L=16384, k=16), 4),       # the splits of 256 KV heads take two steps
    (dict(B=41, L=16000, k=14), 4),
])
def test_noalloc_in_few_even_launches(shape, want_launches):
    """Calls whose unit partials exceed the scratch run as splits, and calls whose split partials do run in as few
    steps as hold them, with the bits of the workspace entry point."""
    print(f"noalloc launches {shape}", flush=True)
    inp = spec.make_inputs(shape, seed=5, dist="randn", device="cuda")
    out = torch.full_like(inp["q"], float("nan"))
    call_noalloc(inp, out)
    want = call_workspace(inp)
    torch.cuda.synchronize()
    assert torch.equal(out.view(torch.int16), want.view(torch.int16))
    assert launches(lambda: call_noalloc(inp, out)) == want_launches
