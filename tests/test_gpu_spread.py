"""Calls that spread their work by the load of the chip give the same bits however it is spread.

The key split (decode and verification up to 64 rows per KV head): a call with few splits deals
units of keys out to all waves and folds them in its combine launch, a call that fills the chip folds them in registers.
Each case runs a batch large enough for the second and every request alone (the first), which must give the same bits,
and checks the batch against the float64 oracle.  A cache of one split takes one launch without a combine, or units with
it: the same bits as well.  Sizes: one tile, ends inside the first unit, block and split and just past them, fewer tiles
than waves, more requests than one scan of the lengths holds, both row-block forms, and 17 to 64 splits to a request
(the combine over units takes 16 at a time)."""
import numpy as np
import pytest
import torch

import oracle
from judge import normalised_error as nerr
from vmk.ops import decode, decode_paged, dsa, prefix, prefix_paged, spec

pytestmark = pytest.mark.gpu

DECODE = [dict(B=70, L=40, L_min=1), dict(B=9, L=2049), dict(B=12, L=4096, L_min=1), dict(B=33, L=1025, L_min=1),
          dict(B=40, L=513, Hq=8, Hkv=1), dict(B=33, L=1280, L_min=1), dict(B=33, L=1281, L_min=1),
          dict(B=33, L=2048, L_min=1, dtype="bf16"), dict(B=9, L=2500, L_min=1, Hq=64, Hkv=8, dtype="bf16"),
          dict(B=24, L=6000, L_min=1, Hq=48, Hkv=2), dict(B=5, L=40000, L_min=32769, Hq=8, Hkv=1),
          dict(B=3, L=131072, L_min=34000, Hq=8, Hkv=1, dtype="bf16"), dict(B=4, L=34816, L_min=1, Hq=24, Hkv=1)]
PAGED = [dict(B=20, L=1504, L_min=1, ps=32, dtype="bf16"), dict(B=20, L=2048, L_min=1, ps=64, layout="NHD"),
         dict(B=10, L=2100, L_min=1, ps=64), dict(B=10, L=4100, L_min=1, ps=32, layout="NHD", dtype="bf16"),
         dict(B=3, L=67584, L_min=33000, Hq=8, Hkv=1, ps=64)]
SPEC = [dict(B=9, L=2049, k=8), dict(B=5, L=8300, k=5), dict(B=10, L=4200, k=16), dict(B=9, L=300, k=11, Hq=8, Hkv=2),
        dict(B=9, L=640, k=16), dict(B=9, L=1500, k=16, dtype="bf16"), dict(B=12, L=2048, k=7),
        dict(B=6, L=16500, k=2), dict(B=5, L=20000, k=9), dict(B=8, L=70000, k=16, Hq=4, Hkv=1),
        dict(B=4, L=40000, k=3, Hq=8, Hkv=1, dtype="bf16")]
# Shared prefix as single waves (two rounds of the mixed launch, up to 96 rows per KV head) and each request alone,
# which is not: one, two and three row blocks, the last row, tile and chunk partly filled, suffixes of no rows, of fewer
# tiles than waves and of the most rows, one and eight rows per KV head; and full suffixes of one round, which stay
# mixed (N = 16 of 2 rows after 2048 keys) or not (after 8192).
PREFIX = [dict(N=24, P=8000, S=1000, S_min=0), dict(N=9, P=8191, S=1025, S_min=1), dict(N=13, P=7409, S=34),
          dict(N=12, P=4100, S=500, S_min=0, Hq=64, dtype="bf16"), dict(N=20, P=5000, S=2048, S_min=1),
          dict(N=9, P=4100, S=300, S_min=0, Hq=32, Hkv=32), dict(N=16, P=2048, S=1024, Hq=32, Hkv=16),
          dict(N=16, P=8192, S=1024, Hq=32, Hkv=16)]
PREFIX_PAGED = [dict(N=24, P=8192, S=1000, S_min=0, ps=64, dtype="bf16"),
                dict(N=11, P=4704, S=700, S_min=0, ps=32, layout="NHD", Hq=64, absent=2),
                dict(N=20, P=5024, S=2048, S_min=1, ps=32, dtype="bf16")]
# DSA decode of batches on indexer workgroups of 1024 positions and each request alone on 256: the last workgroup and
# tile partly filled, one position past the selection, and the longest request that takes the small ones.
DSA = [dict(B=30, L=2049), dict(B=9, L=8100, dtype="bf16"), dict(B=5, L=16384), dict(B=17, L=4097)]


def same_bits(a, b):
    return torch.equal(a.view(torch.int16), b.view(torch.int16))


def check(out, ref):
    torch.cuda.synchronize()
    em, _ = nerr(out.float().cpu().numpy().astype(np.float64), ref)
    print(f"  err max {em:.3e}", flush=True)
    # 16-bit results of values below 5: half a unit of the last place is 2^-9 of the value in bf16, 2^-12 in fp16; P and
    # the partials round at the same precision, so the sum stays within four of them.
    assert em <= (4 * 2.0 ** -9 if out.dtype == torch.bfloat16 else 4 * 2.0 ** -12)


@pytest.mark.parametrize("shape", DECODE)
def test_decode_batch_equals_requests_alone(shape):
    import vmk
    print(f"decode {shape}", flush=True)
    inp = decode.make_inputs(shape, seed=41, device="cuda")
    out = vmk.decode(**inp)
    for i in range(shape["B"]):
        assert same_bits(vmk.decode(**decode.row_inputs(inp, i))[0], out[i]), i
    check(out, oracle.decode.ref64(**inp))


@pytest.mark.parametrize("shape", PAGED)
def test_paged_decode_batch_equals_requests_alone(shape):
    import vmk
    print(f"decode_paged {shape}", flush=True)
    inp = decode_paged.make_inputs(shape, seed=42, device="cuda")
    out = vmk.decode_paged(**inp)
    for i in range(shape["B"]):
        assert same_bits(vmk.decode_paged(**decode_paged.row_inputs(inp, i))[0], out[i]), i
    check(out, oracle.decode_paged.ref64(**inp))


@pytest.mark.parametrize("shape", SPEC)
def test_verify_batch_equals_requests_alone(shape):
    import spec_mi355x
    print(f"spec {shape}", flush=True)
    inp = spec.make_inputs(shape, seed=43, dist="chain", device="cuda")
    out = spec_mi355x.kernel(**inp)
    for i in range(shape["B"]):
        assert same_bits(spec_mi355x.kernel(**spec.row_inputs(inp, i))[0], out[i]), i
    check(out, oracle.spec.ref64(**inp))


@pytest.mark.parametrize("shape", PREFIX)
def test_prefix_batch_equals_requests_alone(shape):
    import vmk
    print(f"prefix {shape}", flush=True)
    inp = prefix.make_inputs(shape, seed=44, device="cuda")
    out = vmk.prefix_decode(**inp)
    for i in range(shape["N"]):
        assert same_bits(vmk.prefix_decode(**prefix.row_inputs(inp, i))[0], out[i]), i
    check(out, oracle.prefix.ref64(**inp))


@pytest.mark.parametrize("shape", PREFIX_PAGED)
def test_paged_prefix_batch_equals_requests_alone(shape):
    import vmk
    print(f"prefix_paged {shape}", flush=True)
    inp = prefix_paged.make_inputs(shape, seed=45, device="cuda")
    out = vmk.prefix_decode_paged(**inp)
    for i in range(shape["N"]):
        assert same_bits(vmk.prefix_decode_paged(**prefix_paged.row_inputs(inp, i))[0], out[i]), i
    check(out, oracle.prefix_paged.ref64(**inp))


@pytest.mark.parametrize("shape", DSA)
def test_dsa_batch_equals_requests_alone(shape):
    import vmk
    print(f"dsa {shape}", flush=True)
    inp = dsa.make_inputs(shape, seed=46, dist="ragged", device="cuda")

    def run(x):
        B = x["q"].shape[0]
        idx = torch.full((B, 2048), -1, dtype=torch.int32, device="cuda")
        cnt = torch.full((B,), -7, dtype=torch.int32, device="cuda")
        out = vmk.dsa_decode(x["q"], x["kv"], x["iq"], x["ik"], x["w"], x["lens"], idx=idx, cnt=cnt)
        return out, idx, cnt

    out, idx, cnt = run(inp)
    scores = vmk.dsa_indexer(inp["iq"], inp["ik"], inp["w"], inp["lens"])
    for i in range(shape["B"]):
        x = {k: None if v is None else v[i:i + 1].contiguous() for k, v in inp.items()}
        o, ix, c = run(x)
        assert same_bits(o[0], out[i]) and torch.equal(ix[0], idx[i]) and torch.equal(c[0], cnt[i]), i
        n = int(x["lens"][0])
        s = vmk.dsa_indexer(x["iq"], x["ik"], x["w"], x["lens"])
        assert torch.equal(s[0, :n].view(torch.int32), scores[i, :n].view(torch.int32)), i
