"""The prefill GEMM1's row classes (how deep its operand rings run by the rows of an item)
at their edges: experts with exactly the row counts where a 16-row block, a class (40 / 41,
144 / 145) or a 256-row tile begins or ends, and where experts of one tile and of several
share a call, checked row by row against the fp32 oracle, and
pair 8/5 from T = 560 on, where this kernel stands in for the token-sharing GEMM1, against
pair 7/5, whose C goes through fp16 and the conversion: bit-identical outputs.  The GEMM2's row classes
(T <= 1200) against the two-stage kernel of larger calls, bit-identical too."""
import pytest
import torch

from conftest import oracle, pkg
from gpu_common import config_inputs, first_tokens, note

pytestmark = pytest.mark.gpu

EDGES = (1, 15, 16, 17, 32, 33, 39, 40, 41, 47, 48, 49, 64, 65, 127, 128, 129, 143, 144, 145,
         0, 160, 161, 239, 240, 241, 255, 256, 257, 0, 296, 397)
# one-tile experts (weights loaded non-temporal up to T = 2560) among experts of several tiles
MIXED = (1, 257, 0, 300, 256, 513, 41, 145) + (0,) * 23 + (17,)   # 1530 tokens
SMALL = (1, 16, 17, 0, 40, 41, 64, 65, 128, 0, 129, 144, 145, 0, 64)   # 854 tokens

# the GEMM2's classes (24 / 25, 64 / 65) and 128-row tiles, experts of one tile and of several
GEMM2 = (24, 25, 64, 65, 128, 129, 1, 16, 17, 0, 32, 33, 48, 49, 0, 23, 63, 127, 257)   # 1101 tokens

# the token-sharing GEMM1's 64-row tiles: experts of one tile and of two (weights loaded
# non-temporal), of three and four (not), and light ones next to them
TOKEN_SHARING = (64, 63, 65, 1, 0, 130, 193, 0, 16, 17)   # 549 tokens


def _inputs(counts):
    """One local expert per token, counts[e] tokens for local expert e in a shuffled order;
    the other seven picks are experts of groups 1 .. 3 (not local at offset 0)."""
    wl = pkg("workloads")
    T = sum(counts)
    g = torch.Generator(device="cuda")
    g.manual_seed(40 + T)
    lg = -6.0 + 0.01 * torch.randn(T, 256, generator=g, device="cuda")
    e = torch.repeat_interleave(torch.arange(len(counts), device="cuda"),
                                torch.tensor(counts, device="cuda"))
    e = e[torch.randperm(T, generator=g, device="cuda")]
    lg[torch.arange(T, device="cuda"), e] = 3.0
    for j in range(7):
        lg[:, 32 * (1 + j % 3) + 5 * j] = 2.0 + 0.1 * j
    hs, sc = wl.quantize_rows_128(torch.randn(T, 7168, generator=g, device="cuda").to(torch.bfloat16))
    d = dict(config_inputs(3))
    d.update(routing_logits=lg, routing_bias=torch.zeros(256, dtype=torch.bfloat16, device="cuda"),
             hidden_states=hs, hidden_states_scale=sc, local_expert_offset=0,
             output=torch.empty(T, 7168, dtype=torch.bfloat16, device="cuda"))
    return d, T


def _run(d, T, flags):
    k = pkg("kernel")
    wl = pkg("workloads")
    lay = k.workspace_layout(T, flags)
    ws = torch.full((lay.total,), 255, dtype=torch.uint8, device="cuda")   # fp8 / fp16 NaN
    out = torch.full_like(d["output"], float("nan"))
    k.forward(*wl.as_args({**d, "output": out}), workspace=ws, flags=flags)
    torch.cuda.synchronize()
    assert not torch.isnan(out).any()
    return lay, ws, out


@pytest.mark.parametrize("counts,scales", [(EDGES, "gathered"), (EDGES, "by token"), (MIXED, "gathered")],
                         ids=["gathered", "by token", "one-tile among larger"])
def test_row_counts_at_the_class_edges(counts, scales):
    k = pkg("kernel")
    o = oracle()
    d, T = _inputs(counts)
    note(f"[gpu] row classes T={T} scales {scales}")
    lay, ws, _ = _run(d, T, k.FLAG_ROW_SCALES_OFF if scales == "by token" else 0)
    assert lay.tile_m == 256
    R = T * 8
    off = ws[lay.meta:lay.meta + 33 * 4].view(torch.int32).cpu().tolist()
    assert [off[e + 1] - off[e] for e in range(32)] == list(counts)
    stok = ws[lay.sorted_tokens:lay.sorted_tokens + off[32] * 4].view(torch.int32).cpu().tolist()
    hi = ws[lay.intermediate:lay.intermediate + R * 2048].view(R, 2048)
    lo = ws[lay.intermediate + R * 2048:lay.intermediate + 2 * R * 2048].view(R, 2048)
    sc = ws[lay.intermediate_scales:lay.intermediate_scales + 16 * R * 4].view(torch.float32).view(16, R)
    for e, n in enumerate(counts):
        # first, last and block- or tile-edge rows of the expert
        rows = sorted({off[e] + r for r in (0, 15, 16, 127, 128, 255, 256, n // 2, n - 1) if 0 <= r < n})
        if not rows:
            continue
        idx = torch.tensor(rows, device="cuda")
        got = o.hilo_join(hi[idx].cpu(), lo[idx].cpu(), sc[:, idx].t().contiguous().cpu())
        ref = o.swiglu_rows(d["hidden_states"], d["hidden_states_scale"], d["gemm1_weights"],
                            d["gemm1_weights_scale"], e, [stok[r] for r in rows])
        # hi + lo/16 of e4m3 parts holds a value to 2^-8 of itself or of its block's maximum
        # (lo's own granule); twice that, for the fp32 sums' order
        bmax = ref.view(-1, 16, 128).abs().amax(dim=2).repeat_interleave(128, dim=1)
        err = (got - ref).abs()
        assert (err <= ref.abs() * 2.0 ** -7 + bmax * 2.0 ** -10).all(), (e, n, float(err.max()))


def test_pair_8_5_is_bit_identical_to_7_5():
    k = pkg("kernel")
    d, T = _inputs(SMALL)
    assert T >= 560
    note(f"[gpu] pair 8/5 by row classes T={T}")
    _, _, ref = _run(d, T, k.plan_flags(7, 5))
    for flags in (0, k.plan_flags(8, 5), k.FLAG_LIST_ORDER, k.FLAG_ROW_SCALES_OFF, k.FLAG_ROW_SCALES_ON):
        _, _, out = _run(d, T, flags)
        assert torch.equal(out.view(torch.int16), ref.view(torch.int16)), flags


@pytest.mark.parametrize("pair", [(0, 0), (4, 5), (7, 5)], ids=["default", "4/5", "7/5"])
def test_gemm2_classes_are_bit_identical_to_the_two_stage_kernel(pair):
    """The same tokens in a call of more than 1200: an output row does not depend on the
    call's other tokens, and there GEMM2 runs its two-stage kernel."""
    k = pkg("kernel")
    d, T = _inputs(GEMM2)
    assert T <= 1200 < T + 200 <= 1344
    note(f"[gpu] GEMM2 row classes T={T} pair {pair}")
    flags = k.plan_flags(*pair) if pair[0] else 0
    big = dict(d, output=torch.empty(T + 200, 7168, dtype=torch.bfloat16, device="cuda"))
    for name in ("routing_logits", "hidden_states"):
        big[name] = torch.cat([d[name].view(torch.uint8)] * 2)[:T + 200].view(d[name].dtype).contiguous()
    big["hidden_states_scale"] = torch.cat([d["hidden_states_scale"]] * 2, dim=1)[:, :T + 200].contiguous()
    _, _, out = _run(d, T, flags)
    _, _, ref = _run(big, T + 200, flags)
    assert torch.equal(out.view(torch.int16), ref[:T].view(torch.int16))


@pytest.mark.parametrize("T", [560, 700, 1024, 1344, None], ids=["560", "700", "1024", "1344", "class edges"])
def test_values_beyond_fp16_match_the_converted_form(T):
    """Every third token 2^10 times larger, so that C leaves the fp16 range in some rows, and
    in some 16-column groups beside values that stay inside it: the rows in use are those of
    the token-sharing GEMM1 and the conversion (pair 7/5) bit for bit, the C flag (meta[35])
    and the row flag are raised, and a call on normal inputs afterwards leaves both at zero
    (the LDS rows past a tile then still hold large values)."""
    k = pkg("kernel")
    if T is None:
        d, T = _inputs(SMALL)
    else:
        d = first_tokens(config_inputs(3), T)
    note(f"[gpu] beyond fp16 by row classes T={T}")
    scale = d["hidden_states_scale"].clone()
    scale[:, ::3] *= 1024.0
    big = dict(d, hidden_states_scale=scale)

    def used(lay, ws):
        R = T * 8
        na = int(ws[lay.meta + 32 * 4:lay.meta + 33 * 4].view(torch.int32).item())
        c = ws[lay.intermediate:lay.intermediate + 2 * R * 2048].view(2, R, 2048)[:, :na]
        s = ws[lay.intermediate_scales:lay.intermediate_scales + 16 * R * 4].view(torch.int32).view(16, R)[:, :na]
        flags = ws[lay.meta + 35 * 4:lay.meta + 37 * 4].view(torch.int32).cpu().tolist()
        return c, s, flags

    lay, ws, ref = _run(big, T, k.plan_flags(7, 5))
    ref_c, ref_s, flags = used(lay, ws)
    assert flags == [1, 1]
    for fl in (0, k.plan_flags(8, 5), k.FLAG_LIST_ORDER, k.FLAG_ROW_SCALES_OFF):
        lay, ws, out = _run(big, T, fl)
        c, s, flags = used(lay, ws)
        assert flags == [1, 1], fl
        assert torch.equal(c, ref_c) and torch.equal(s, ref_s), fl
        assert torch.equal(out.view(torch.int16), ref.view(torch.int16)), fl
    lay, ws, out = _run(d, T, 0)
    assert used(lay, ws)[2] == [0, 0]
    _, _, ref = _run(d, T, k.plan_flags(7, 5))
    assert torch.equal(out.view(torch.int16), ref.view(torch.int16))


@pytest.mark.parametrize("pair", [(8, 7), (7, 7)], ids=["8/7", "7/7"])
def test_token_sharing_tiles_match_oracle(pair):
    k = pkg("kernel")
    o = oracle()
    d, T = _inputs(TOKEN_SHARING)
    assert 200 <= T <= 559
    note(f"[gpu] token-sharing tiles T={T} pair {pair}")
    lay, ws, _ = _run(d, T, k.plan_flags(*pair))
    assert lay.tile_m == 64 and lay.intermediate_format == 0
    R = T * 8
    off = ws[lay.meta:lay.meta + 33 * 4].view(torch.int32).cpu().tolist()
    assert [off[e + 1] - off[e] for e in range(len(TOKEN_SHARING))] == list(TOKEN_SHARING)
    stok = ws[lay.sorted_tokens:lay.sorted_tokens + off[32] * 4].view(torch.int32).cpu().tolist()
    f16 = ws[lay.intermediate + 2 * R * 2048:lay.intermediate + 4 * R * 2048].view(torch.float16).view(R, 2048)
    for e, n in enumerate(TOKEN_SHARING):
        rows = sorted({off[e] + r for r in (0, 15, 16, 47, 48, 63, 64, 127, 128, 191, 192, n - 1) if 0 <= r < n})
        if not rows:
            continue
        got = f16[torch.tensor(rows, device="cuda")].float().cpu()
        ref = o.swiglu_rows(d["hidden_states"], d["hidden_states_scale"], d["gemm1_weights"],
                            d["gemm1_weights_scale"], e, [stok[r] for r in rows])
        # fp16 rounds to 2^-11 of a value; twice that, and 2^-12 of the row's 128-column
        # maximum for the fp32 sums' order
        bmax = ref.view(-1, 16, 128).abs().amax(dim=2).repeat_interleave(128, dim=1)
        err = (got - ref).abs()
        assert (err <= ref.abs() * 2.0 ** -10 + bmax * 2.0 ** -12).all(), (e, n, float(err.max()))


@pytest.mark.parametrize("T", [27000, 32768], ids=["in the item table", "past the item table"])
def test_many_rounds_of_items(T):
    """Every route local: 8 T rows.  The prefill GEMM1 ranks up to 56 rounds of items per
    workgroup (T = 27000: 54); beyond (T = 32768: 66) it takes them in list order and resolves
    those past its table one by one.  An output row does not depend on the call's other tokens:
    the first and last tokens equal those of calls of their own."""
    k = pkg("kernel")
    wl = pkg("workloads")
    cfg = wl.Config("all_local", T, 0, hot_local_experts=tuple(range(32)), seed=20261111)
    d = dict(config_inputs(4))
    d.update(wl.make_activations(cfg, device="cuda"))
    d["output"] = torch.empty(T, 7168, dtype=torch.bfloat16, device="cuda")
    note(f"[gpu] rounds of items, all local T={T}")
    lay, ws, out = _run(d, T, 0)
    off = ws[lay.meta:lay.meta + 33 * 4].view(torch.int32).cpu().tolist()
    items = 16 * sum((b - a + 255) // 256 for a, b in zip(off, off[1:]))
    assert off[32] == 8 * T and (items > 56 * 256) == (T == 32768)
    if T == 27000:
        _, _, ref = _run(d, T, k.FLAG_LIST_ORDER)
        assert torch.equal(out.view(torch.int16), ref.view(torch.int16))
        return
    del ws
    for part in (slice(0, 1700), slice(T - 1700, T)):
        p = dict(d, routing_logits=d["routing_logits"][part].contiguous(),
                 hidden_states=d["hidden_states"][part].contiguous(),
                 hidden_states_scale=d["hidden_states_scale"][:, part].contiguous(),
                 output=torch.empty(1700, 7168, dtype=torch.bfloat16, device="cuda"))
        _, _, ref = _run(p, 1700, 0)
        assert torch.equal(out[part].view(torch.int16), ref.view(torch.int16))
