"""A request's bits depend on its own rows, length and keys, not on how many positions its cache could hold.

The same requests decode from caches of several capacities (positions past a request's length hold other values) and
must give the same bits: around the capacity of one split, where a longer cache adds a combine launch or deals the keys
out as units, and around the lengths at which groups of many rows take larger splits."""
import pytest
import torch

import oracle
from judge import normalised_error as nerr

pytestmark = pytest.mark.gpu

# (Hq, Hkv, dtype, lengths, capacities): 4 rows a group on both sides of one split, in batches that take splits and in
# single requests that take units; 32 and 64 rows past 16384 positions; 24 rows past 2^20.
CASES = [
    (32, 8, "bf16", [1, 700, 2047, 2048], [2048, 2049, 9000, 40000]),
    (32, 8, "bf16", [1999], [1999, 2048, 2049, 4096, 65536]),
    (32, 8, "fp16", [37, 1500], [1500, 2048, 5000]),
    (32, 8, "bf16", [64 * i + 5 for i in range(34)], [2117, 4000]),
    (64, 2, "bf16", [3000, 16384, 12345], [16384, 16385, 40000]),
    (64, 1, "fp16", [5, 2048, 16001], [16001, 33000, 70000]),
    (64, 1, "bf16", [16385, 20000, 900], [20000, 66000]),
    (24, 1, "fp16", [30001, 2048], [30001, (1 << 20) + 64]),
]


def same_bits(a, b):
    return torch.equal(a.view(torch.int16), b.view(torch.int16))


@pytest.mark.parametrize("Hq,Hkv,dtype,lens,caps", CASES)
def test_decode_bits_do_not_depend_on_the_capacity(Hq, Hkv, dtype, lens, caps):
    import vmk
    print(f"capacity {Hq}/{Hkv} {dtype} {lens[:4]} {caps}", flush=True)
    dt = {"fp16": torch.float16, "bf16": torch.bfloat16}[dtype]
    g = torch.Generator(device="cuda").manual_seed(17)

    def r(*shape):
        return torch.randn(shape, generator=g, device="cuda").to(dt)
    B, n = len(lens), max(lens)
    q, k0, v0 = r(B, Hq, 128), r(B, Hkv, n, 128), r(B, Hkv, n, 128)
    ln = torch.tensor(lens, dtype=torch.int32, device="cuda")
    outs = []
    for cap in caps:
        k, v = r(1, 1, cap, 128).repeat(B, Hkv, 1, 1), r(1, 1, cap, 128).repeat(B, Hkv, 1, 1)
        k[:, :, :n], v[:, :, :n] = k0, v0
        outs.append(vmk.decode(q, k, v, lens=ln))
        assert same_bits(outs[-1], outs[0]), (cap, int((outs[-1] != outs[0]).sum()))
    if caps[-1] < 1 << 20:
        ref = oracle.decode.ref64(q=q, k=k0, v=v0, lens=ln)
        em, _ = nerr(outs[0].double().cpu().numpy(), ref)
        # Half a unit of the last place of a 16-bit result, and as much again for P, the partials and their sum.
        assert em <= 4 * (2.0 ** -9 if dtype == "bf16" else 2.0 ** -12)


@pytest.mark.parametrize("dtype,lens", [("bf16", [1, 333, 2048]), ("fp16", [2000])])
def test_paged_decode_bits_do_not_depend_on_the_table_length(dtype, lens):
    import vmk
    dt = {"fp16": torch.float16, "bf16": torch.bfloat16}[dtype]
    g = torch.Generator(device="cuda").manual_seed(18)
    ps, B = 64, len(lens)
    pool_k, pool_v = (torch.randn((4 * 32 + 9, 8, ps, 128), generator=g, device="cuda").to(dt) for _ in range(2))
    q = torch.randn((B, 32, 128), generator=g, device="cuda").to(dt)
    ln = torch.tensor(lens, dtype=torch.int32, device="cuda")
    table = torch.randperm(B * 32, generator=torch.Generator().manual_seed(3)).to(torch.int32).view(B, 32).cuda()
    first = vmk.decode_paged(q, pool_k, pool_v, table, lens=ln)
    for more in (1, 33, 600):
        longer = torch.cat([table, torch.full((B, more), -1, dtype=torch.int32, device="cuda")], 1).contiguous()
        out = vmk.decode_paged(q, pool_k, pool_v, longer, lens=ln)
        assert same_bits(out, first), (more, int((out != first).sum()))
