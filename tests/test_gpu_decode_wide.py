"""The wide matrix-core decode (17 to 128 rows) against the fp32 reconstruct + matmul of the oracle.

Bounds (relative L2): fp16 operands and outputs each round by at most 2^-11 of their value, fp16(x h) and y make
2^-10; S_group adds the rounding of the scaled table vector and of the oracle's W; a bf16 output rounds by 2^-9."""

import pytest
import torch

from eptq_amd.kernels import decode_workspace, linear_forward_multi
from eptq_amd.kernels.linear import EPTQLinear, EPTQMultiLinear
from eptq_amd.synthetic import make_layer
from oracle.matvec import linear_ref, rel_l2

from _util import layer_np, table

pytestmark = pytest.mark.gpu


def _layer(out, inp, seed, p, qb=None):
    qd = make_layer(out, inp, seed=seed, percmask=p, bias=True, qb_size=qb)
    return qd, EPTQLinear.from_quantized_data(qd, torch.from_numpy(table("e8_d4", 1.75)), "e8_d4").to("cuda:0")


def _ref(qd, x):
    n = layer_np(qd)
    return linear_ref(x.float().cpu().numpy(), n["Q"], n["g"], n["h"], n["O"], table("e8_d4", 1.75), "e8_d4",
                      bias=qd.bias.float().numpy(), S_group=n["S_group"])


# Edges: one and several row tiles (a ragged last one), column counts off the blocks of 32 and 64, row counts at the
# edges of the groups of 16 and 64, more critical blocks than the LDS stage holds, group sizes, both types.
@pytest.mark.parametrize("out,inp,T,p,qb,dt", [
    (8, 8, 17, 0.0, None, torch.float16),
    (72, 200, 31, 0.02, None, torch.float16),
    (520, 1096, 33, 0.01, None, torch.float16),
    (1024, 4104, 48, 0.002, None, torch.float16),
    (1024, 4096, 64, 0.01, 128, torch.float16),
    (256, 2048, 65, 0.6, None, torch.float16),
    (256, 11008, 96, 0.3, 64, torch.bfloat16),
    (4096, 1024, 112, 0.002, None, torch.bfloat16),
    (1536, 768, 128, 0.002, 128, torch.float16),
])
def test_wide_decode(out, inp, T, p, qb, dt):
    print(f"wide decode {out}x{inp} T={T} p={p} qb={qb} {dt}", flush=True)
    qd, lin = _layer(out, inp, out + inp + T, p, qb)
    x = torch.randn((T, inp), generator=torch.Generator().manual_seed(T)).to(dt)
    ref = _ref(qd, x)
    tol = (2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -10) + (2.0 ** -10 if qb else 0.0)
    ys = []
    for work in (decode_workspace("cuda:0"), None):
        layer = {k: getattr(lin, k) for k in ("Q", "g", "h", "O_vals", "O_col", "O_row_ptr", "bias", "S_group")}
        for _ in range(2):   # the split's counters return to zero
            ys.append(linear_forward_multi([layer], lin._codebook, x.cuda(), work=work))
    for y in ys:
        assert rel_l2(y.float().cpu().numpy(), ref) <= tol
    assert torch.equal(ys[0], ys[1]) and torch.equal(ys[2], ys[3])


def test_wide_decode_rows_do_not_mix():
    """A row of non-finite activations leaves the others alone, also where the last column block ends inside a row."""
    print("wide decode rows", flush=True)
    for inp, T in ((200, 40), (1096, 64), (4104, 20)):
        _, lin = _layer(128, inp, inp, 0.01)
        x = torch.randn((T, inp), generator=torch.Generator().manual_seed(inp)).half().cuda()
        want = lin(x)
        x[1, :40] = float("inf")
        x[1, 64:90] = float("nan")
        got = lin(x)
        keep = torch.arange(T, device="cuda:0") != 1
        assert torch.equal(got[keep], want[keep])
        assert not torch.isfinite(got[1]).any()


@pytest.mark.parametrize("T", [20, 64, 100])
def test_wide_decode_layers_of_one_launch(T):
    """q|k|v of unequal heights in one launch equal the layers alone (another column split of the same sums)."""
    print(f"wide decode multi T={T}", flush=True)
    lins = [_layer(o, 2048, 10 + k, 0.002)[1] for k, o in enumerate((1024, 256, 264))]
    x = torch.randn((T, 2048), generator=torch.Generator().manual_seed(T)).half().cuda()
    y = EPTQMultiLinear(lins)(x)
    one = torch.cat([l(x) for l in lins], dim=-1)
    assert rel_l2(y.float().cpu().numpy(), one.float().cpu().numpy()) <= 2.0 ** -10
