"""Ragged decode over splits that are dealt to the XCDs in rotation: every split of every group is walked once, whatever
the number of splits and groups.  Batches large enough to run as splits against their requests alone (bit for bit) and
the float64 oracle: 2 to 12 splits, powers of two, odd and even, and groups that start on one, two, four or all XCDs."""
import pytest
import torch

import oracle
from judge import normalised_error as nerr
from vmk.ops import decode, decode_paged

pytestmark = pytest.mark.gpu

SHAPES = [dict(B=33, L=4000, L_min=1, Hq=8, Hkv=1), dict(B=11, L=6000, L_min=1, Hq=12, Hkv=3),
          dict(B=9, L=8192, L_min=1, dtype="bf16"), dict(B=15, L=10000, L_min=1, Hq=16, Hkv=1),
          dict(B=7, L=12000, L_min=1, Hq=10, Hkv=2), dict(B=9, L=16384, L_min=1, Hq=48, Hkv=2),
          dict(B=9, L=24000, L_min=1, Hq=40, Hkv=1, dtype="bf16")]
PAGED = [dict(B=9, L=8192, L_min=1, ps=64, dtype="bf16", layout="NHD"), dict(B=3, L=20480, L_min=1, ps=32)]


def check(op, shape, call):
    print(f"{op.__name__} {shape}", flush=True)
    inp = op.make_inputs(shape, seed=51, device="cuda")
    out = call(**inp)
    for i in range(shape["B"]):
        one = call(**op.row_inputs(inp, i))[0]
        assert torch.equal(one.view(torch.int16), out[i].view(torch.int16)), i
    em, _ = nerr(out.double().cpu().numpy(), getattr(oracle, op.__name__.split(".")[-1]).ref64(**inp))
    # Half a unit of the last place of a 16-bit result, and as much again for P, the partials and their sum.
    assert em <= 4 * (2.0 ** -9 if out.dtype == torch.bfloat16 else 2.0 ** -12)


@pytest.mark.parametrize("shape", SHAPES)
def test_ragged_decode(shape):
    import vmk
    check(decode, shape, vmk.decode)


@pytest.mark.parametrize("shape", PAGED)
def test_ragged_paged_decode(shape):
    import vmk
    check(decode_paged, shape, vmk.decode_paged)
