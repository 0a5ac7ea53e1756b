"""moe_ffn's two products take row tiles of limits of their own: the row-tile
tables in the scratch, where the products' limits differ, against the row counts,
and the result against per-expert calls."""
import numpy as np
import pytest

import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [H.F16, H.BF16])
@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("per,hidden,inter,limits", [
    ([300, 256, 0, 310, 234], 256, 24576, (192, 64)),              # many column tiles and one
    ([1, 65, 128, 129, 192, 0, 193, 257, 320, 513], 4096, 512, (64, 192)),
])
def test_limits_of_both_products(device, dt, bits, per, hidden, inter, limits):
    import torch
    from paddle_amd import _lib
    from paddle_amd.nn import quant as Q

    E, T = len(per), torch.bfloat16 if dt == H.BF16 else torch.float16
    gen = torch.Generator(device="cuda").manual_seed(11)
    algo, wd = "weight_only_int%d" % bits, "int%d" % bits
    q1, s1 = Q.moe_quantize_experts(torch.randn(E, hidden, inter, device="cuda", generator=gen, dtype=T) * 0.02, algo)
    q2, s2 = Q.moe_quantize_experts(torch.randn(E, inter // 2, hidden, device="cuda", generator=gen, dtype=T) * 0.02, algo)
    cum = torch.tensor(np.cumsum(per), dtype=torch.int64, device="cuda")
    rows = sum(per)
    x = torch.randn(rows, hidden, device="cuda", generator=gen).to(T)
    out = torch.full((rows, hidden), 77.0, device="cuda", dtype=T)
    ws_bytes = _lib.lib.wol_moe_ffn_workspace(rows, hidden, inter, E)
    ws = torch.full((ws_bytes,), 0xA5, dtype=torch.uint8, device="cuda")  # dirty on purpose
    _lib.check(_lib.lib.wol_moe_ffn(
        x.data_ptr(), cum.data_ptr(), q1.data_ptr(), None, s1.data_ptr(), q2.data_ptr(), s2.data_ptr(), dt,
        rows, hidden, inter, E, bits, out.data_ptr(), ws.data_ptr(), ws_bytes, torch.cuda.current_stream().cuda_stream))
    # a table has room for 32-row tiles and a header, eight words an entry, and is padded to 256 bytes
    table_bytes = -(-((-(-rows // 32) + E + 1) * 32) // 256) * 256
    for i, limit in enumerate(limits):
        tiles = sum(-(-n // limit) for n in per)
        table = ws[i * table_bytes: i * table_bytes + (tiles + 1) * 32].view(torch.int32).view(-1, 8).cpu().numpy()
        assert table[0, 0] == tiles and table[1:, 2].max() <= limit and table[1:, 2].sum() == rows, (i, table[0, 0], tiles)
    prev = 0
    for e, n in enumerate(per):
        if n:
            fc1 = Q.weight_only_linear(x[prev:prev + n], q1[e], None, s1[e], wd)
            act = (torch.nn.functional.silu(fc1[:, : inter // 2].float()) * fc1[:, inter // 2:].float()).to(T)
            ref = Q.weight_only_linear(act, q2[e], None, s2[e], wd)
            # the same fp32 sums to their order: roundings that fall the other way, each a T ulp (2^-8 bf16, 2^-11 f16),
            # in a few percent of the elements at most
            err = float((out[prev:prev + n].float() - ref.float()).norm() / ref.float().norm())
            assert err <= (2e-3 if dt == H.BF16 else 2.5e-4), (e, n, err)
        prev += n
