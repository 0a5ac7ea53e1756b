"""moe_ffn on weight-only quantised experts (wol_moe_ffn: two grouped GEMM
launches over a device-side row-tile table, swiglu between) against the oracle:
per expert, the oracle's linear (rounded to T, as the reference's fc1 output
is), swiglu in float on those T values, the oracle's linear again
(paddle/phi/kernels/fusion/cutlass/moe_ffn.cu:74-183)."""
import numpy as np
import pytest

import helpers as H

pytestmark = pytest.mark.gpu


def _oracle_moe(oracle, xb, cum, w1b, b1b, w2b, dt, bits):
    rows, hidden = xb.shape
    out = np.zeros((rows, hidden), np.uint16)
    prev = 0
    for e, end in enumerate(cum):
        end = int(end)
        if end > prev:
            c1, s1 = oracle.weight_quantize(w1b[e], dt, bits, -1)
            c2, s2 = oracle.weight_quantize(w2b[e], dt, bits, -1)
            _, fc1 = oracle.linear(xb[prev:end], c1, s1, None if b1b is None else b1b[e], dt, bits, -1)
            _, act = oracle.activation(H.bits_to_f32(fc1, dt), oracle.ACT_SWIGLU, dt)
            _, o = oracle.linear(act, c2, s2, None, dt, bits, -1)
            out[prev:end] = o
        prev = end
    return out


# rows per expert: none, a few, exactly one tile, a tile and a bit, many, none at
# the end (128-row tiles); few rows per expert, with whole and partial tiles
# and one expert far above the average (64-row tiles; 32-row tiles for int4);
# an average of 38 rows (64-row tiles for both bit widths); many rows
ROWS_PER_EXPERT = [[0, 5, 128, 131, 300, 0], [0, 5, 33, 64, 1, 17], [40, 64, 0, 70, 3, 50], [2, 1, 150, 0, 3, 4],
                   [600, 256, 0, 1000, 700, 520]]
# (the first and the last: more than 64 rows on average, tiles of up to 256 rows; the others: tiles of 32 or 64)


@pytest.mark.parametrize("dt", [H.F16, H.BF16])
@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("per,inter", [(p, 512) for p in ROWS_PER_EXPERT] + [(p, 4096) for p in ROWS_PER_EXPERT[1:4]])
def test_moe_ffn_against_oracle(device, oracle, dt, bits, per, inter):
    # inter = 4096 with few rows per expert: the second GEMM (K = 2048) runs with
    # its K cut into runs across workgroups and the kernel that adds them
    import torch
    from paddle_amd.nn import quant as Q

    hidden, E = 256, 6
    cum = np.cumsum(per).astype(np.int64)
    rows = int(cum[-1]) + 3  # three rows that belong to no expert
    rng = np.random.default_rng(5)
    xb = H.make_act(rows, hidden, dt, seed=1)
    w1b = np.stack([H.make_weight(hidden, inter, dt, seed=10 + e) for e in range(E)])
    w2b = np.stack([H.make_weight(inter // 2, hidden, dt, seed=20 + e, std=0.05) for e in range(E)])
    b1b = np.stack([H.make_bias(inter, dt, seed=30 + e) for e in range(E)])
    algo = "weight_only_int8" if bits == 8 else "weight_only_int4"
    w1, s1 = Q.moe_quantize_experts(H.bits_to_torch(w1b, dt, device), algo)
    w2, s2 = Q.moe_quantize_experts(H.bits_to_torch(w2b, dt, device), algo)
    x = H.bits_to_torch(xb, dt, device)
    cnt = torch.from_numpy(cum).to(device)
    for bias in (None, b1b):
        b1 = None if bias is None else H.bits_to_torch(bias, dt, device).reshape(E, 1, inter)
        out = Q.moe_ffn(x, cnt, w1, w2, b1, s1, s2, algo)
        torch.cuda.synchronize()
        got = H.torch_to_bits(out)[: int(cum[-1])]
        want = _oracle_moe(oracle, xb, cum, w1b, bias, w2b, dt, bits)[: int(cum[-1])]
        err = H.rel_l2(H.bits_to_f32(got, dt), H.bits_to_f32(want, dt))
        assert err <= 1e-3, (err, dt, bits, bias is not None)
        # every expert on its own, so that a small expert cannot hide behind a large one
        prev = 0
        for e, end in enumerate(cum):
            if end > prev:
                ee = H.rel_l2(H.bits_to_f32(got[prev:end], dt), H.bits_to_f32(want[prev:end], dt))
                assert ee <= 2e-3, (e, ee)
            prev = int(end)


@pytest.mark.parametrize("rows,E", [(200, 5), (1000, 5), (10000, 150)])  # small tiles; one and three scans of 64 experts
def test_moe_ffn_clamps_running_totals_it_cannot_trust(device, rows, E):
    # token_nums_per_expert comes from the device and is read there only.  Totals
    # that run backwards or past the input's rows are clamped by the table
    # builder to [previous total, rows]: the call computes what it would with
    # the clamped totals and touches no row outside the input.
    import torch
    from paddle_amd.nn import quant as Q

    hidden, inter = 256, 512
    gen = torch.Generator(device="cuda").manual_seed(3)
    w1 = (torch.randn(E, hidden, inter, device="cuda", generator=gen) * 0.02).to(torch.bfloat16)
    w2 = (torch.randn(E, inter // 2, hidden, device="cuda", generator=gen) * 0.02).to(torch.bfloat16)
    q1, s1 = Q.moe_quantize_experts(w1)
    q2, s2 = Q.moe_quantize_experts(w2)
    x = torch.randn(rows, hidden, device="cuda", generator=gen).to(torch.bfloat16)
    if E == 5:
        bad = np.array([70, 30, 150, 10 ** 9, -5])  # backwards, huge, negative
    else:
        bad = np.arange(1, E + 1) * 67
        bad[[3, 63, 64, 100, 127]] = [10, 4500, 5, -7, 9000]  # also in the first and last places of a scan
        bad[-3:] = [2 ** 40, 12, -2 ** 40]
    good = np.maximum.accumulate(np.clip(bad, 0, rows))  # what the clamp makes of it
    bad, good = (torch.from_numpy(v.astype(np.int64)).cuda() for v in (bad, good))
    want = Q.moe_ffn(x, good, q1, q2, None, s1, s2, "weight_only_int8")
    got = Q.moe_ffn(x, bad, q1, q2, None, s1, s2, "weight_only_int8")
    torch.cuda.synchronize()
    assert torch.equal(got, want)


def test_moe_ffn_equals_per_expert_calls(device):
    # the grouped launches against a loop of ordinary calls on each expert's rows
    import torch
    from paddle_amd.nn import quant as Q

    hidden, inter, E = 512, 1024, 4
    gen = torch.Generator(device="cuda").manual_seed(9)
    w1 = (torch.randn(E, hidden, inter, device="cuda", generator=gen) * 0.02).to(torch.bfloat16)
    w2 = (torch.randn(E, inter // 2, hidden, device="cuda", generator=gen) * 0.02).to(torch.bfloat16)
    q1, s1 = Q.moe_quantize_experts(w1)
    q2, s2 = Q.moe_quantize_experts(w2)
    per = [40, 0, 260, 17]
    cum = torch.tensor(np.cumsum(per), dtype=torch.int64, device="cuda")
    x = torch.randn(sum(per), hidden, device="cuda", generator=gen).to(torch.bfloat16)
    out = Q.moe_ffn(x, cum, q1, q2, None, s1, s2, "weight_only_int8")
    prev = 0
    for e, n in enumerate(per):
        if n:
            fc1 = Q.weight_only_linear(x[prev:prev + n], q1[e], None, s1[e], "int8")
            act = (torch.nn.functional.silu(fc1[:, : inter // 2].float()) * fc1[:, inter // 2:].float()).to(torch.bfloat16)
            ref = Q.weight_only_linear(act, q2[e], None, s2[e], "int8")
            err = float((out[prev:prev + n].float() - ref.float()).norm() / ref.float().norm())
            assert err <= 2e-3, (e, err)
        prev += n
    with pytest.raises(ValueError):
        Q.moe_ffn(x, cum, q1, q2, None, s1, s2, "None")
    with pytest.raises(ValueError):
        Q.moe_ffn(x, cum.int(), q1, q2, None, s1, s2, "weight_only_int8")


ANY_LOAD = [1, 63, 64, 65, 128, 129, 192, 0, 193, 256, 257, 320, 511, 513]


@pytest.mark.parametrize("dt", [H.F16, H.BF16])
@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("per,hidden,inter,limit", [
    (ANY_LOAD, 256, 512, 64),      # few column tiles: the lowest tiles; second product on 128-column tiles
    (ANY_LOAD, 4096, 512, 64),     # second product on 256-column tiles
    (ANY_LOAD, 1152, 2048, 128),   # 128-column tiles, an odd number of them
    (ANY_LOAD, 4224, 2048, 128),   # 256-column tiles, the last of 128 columns
    ([192, 190, 129, 150, 0, 161, 192, 130, 175], 4224, 8192, 192),  # one tile an expert fills one round
    ([256, 193, 250, 224, 0, 256, 240, 200, 255], 4224, 8192, 256),
])
def test_moe_ffn_tile_heights(device, dt, bits, per, hidden, inter, limit):
    # experts with many rows take row tiles of one to four 64-row units, up to a limit that the number of tiles
    # decides: row counts on both sides of every unit and of one and two whole tiles, an expert without rows.
    # Rows behind the last expert's are left alone.
    import torch
    from paddle_amd import _lib
    from paddle_amd.nn import quant as Q

    E, T = len(per), torch.bfloat16 if dt == H.BF16 else torch.float16
    gen = torch.Generator(device="cuda").manual_seed(11)
    algo, wd = ("weight_only_int8", "int8") if bits == 8 else ("weight_only_int4", "int4")
    q1, s1 = Q.moe_quantize_experts(torch.randn(E, hidden, inter, device="cuda", generator=gen, dtype=T) * 0.02, algo)
    q2, s2 = Q.moe_quantize_experts(torch.randn(E, inter // 2, hidden, device="cuda", generator=gen, dtype=T) * 0.02, algo)
    b1 = torch.randn(E, inter, device="cuda", generator=gen).to(T)
    cum = torch.tensor(np.cumsum(per), dtype=torch.int64, device="cuda")
    rows = sum(per) + 5
    x = torch.randn(rows, hidden, device="cuda", generator=gen).to(T)
    out = torch.full((rows, hidden), 77.0, device="cuda", dtype=T)
    ws_bytes = _lib.lib.wol_moe_ffn_workspace(rows, hidden, inter, E)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device="cuda")
    _lib.check(_lib.lib.wol_moe_ffn(
        x.data_ptr(), cum.data_ptr(), q1.data_ptr(), b1.data_ptr(), s1.data_ptr(), q2.data_ptr(), s2.data_ptr(), dt,
        rows, hidden, inter, E, bits, out.data_ptr(), ws.data_ptr(), ws_bytes, torch.cuda.current_stream().cuda_stream))
    # the row-tile table at the start of the scratch, eight words an entry: the number of tiles in front, then
    # each tile's expert, first row and rows
    tiles = sum(-(-n // limit) for n in per)
    table = ws[: (tiles + 1) * 32].view(torch.int32).view(-1, 8).cpu().numpy()
    assert table[0, 0] == tiles and table[1:, 2].max() <= limit
    assert table[1:, 2].sum() == sum(per)
    assert torch.equal(Q.moe_ffn(x, cum, q1, q2, b1, s1, s2, algo)[: sum(per)], out[: sum(per)])
    assert bool((out[sum(per):] == 77.0).all())
    prev = 0
    for e, n in enumerate(per):
        if n:
            fc1 = Q.weight_only_linear(x[prev:prev + n], q1[e], b1[e], s1[e], wd)
            act = (torch.nn.functional.silu(fc1[:, : inter // 2].float()) * fc1[:, inter // 2:].float()).to(T)
            ref = Q.weight_only_linear(act, q2[e], None, s2[e], wd)
            # same fp32 sums to their order, rounded to T in the same places: only roundings that fall the other
            # way differ, each by a T ulp (2^-8 bf16, 2^-11 f16), in a few percent of the elements at most
            err = float((out[prev:prev + n].float() - ref.float()).norm() / ref.float().norm())
            assert err <= (2e-3 if dt == H.BF16 else 2.5e-4), (e, n, err)
        prev += n
