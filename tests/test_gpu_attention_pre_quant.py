"""GPU parity: GLM-4.5 attention_pre_quant (HIP, through the C ABI) against the CPU oracle.

Bar.  The reference's own test compares all four outputs with rtol 0.0078125 / atol 1e-4
(glm_attention_pre_quant.py:620-631).  The kernels keep every rounding point of the operator and the projection is
exact integer arithmetic; what differs from the oracle is the order of the fp32 sums of squares of the three norms.
In the first norm that now and then moves a value across a bf16 rounding boundary and then, more rarely, an int8 value
of the quantised row by one step - which shifts every output of that token by up to 128 dequantisation steps, far
beyond the reference's tolerance for the outputs that happen to be small.  The quantised row is an intermediate the
operator does not return, so the tests call the C ABI with a workspace of their own and read it there:
  residual_res                         bit-equal to the oracle
  quantised row                        within one step of the oracle's everywhere, equal in at least 99.9 % of the places
  value                                bit-equal to the oracle's stages run on the product's own quantised row
  query, key                           against the same: inside the reference's tolerance except for at most 0.1 % of
                                       the elements (a head norm's sum order, through a bf16 boundary, into a rotary
                                       pair that cancels), none beyond 3 x the tolerance taken on the magnitude of
                                       its rotary pair, at least 98 % bit-equal
  tokens whose quantised row is equal  the same bars against the oracle end to end
"""
import ctypes

import pytest
import torch

from oracle import attention_pre_quant as op

pytestmark = pytest.mark.gpu

NAMES = ["hidden_states", "residual", "input_layernorm_weight", "input_layernorm_bias", "atten_qkv_input_scale_reciprocal",
         "atten_qkv_input_offset", "atten_qkv_weight", "atten_qkv_quant_bias", "atten_qkv_deq_scale", "atten_q_norm_weight",
         "atten_q_norm_bias", "atten_k_norm_weight", "atten_k_norm_bias", "cos", "sin"]


def outputs(case, dev):
    t, h = case["hidden_states"].shape
    bf = torch.bfloat16
    # outputs start as NaN: an element the kernels leave out shows
    return {"query": torch.full((t, case["q_size"]), float("nan"), dtype=bf, device=dev),
            "key": torch.full((t, case["kv_size"]), float("nan"), dtype=bf, device=dev),
            "value": torch.full((t, case["kv_size"]), float("nan"), dtype=bf, device=dev),
            "residual_res": torch.full((t, h), float("nan"), dtype=bf, device=dev)}


def run_operator(case, dev):
    """Through the Python operator (which sizes and allocates the workspace itself)."""
    from pypto_amd.glm_v4_5 import glm_attention_pre_quant as impl
    out = outputs(case, dev)
    impl.attention_pre_quant(*[case[k].to(dev) for k in NAMES], out["query"], out["key"], out["value"],
                             out["residual_res"])
    torch.cuda.synchronize()
    return {k: v.cpu() for k, v in out.items()}


def run(case, dev):
    """Through the C ABI with a workspace of the test's own, whose head holds the quantised rows [t, h] afterwards."""
    from pypto_amd import _runtime
    lib = _runtime.load_library()
    t, h = case["hidden_states"].shape
    out = outputs(case, dev)
    tensors = [case[k].to(dev) for k in NAMES] + [out["query"], out["key"], out["value"], out["residual_res"]]
    descs = _runtime.describe(tensors)
    p = _runtime.AttentionPreQuantParams(op.EPS)
    n = lib.pto_attention_pre_quant_workspace(descs, 19, ctypes.byref(p))
    assert n > 0 or t == 0, lib.pto_last_error().decode()
    ws = torch.full((max(n, 1),), 0x55, dtype=torch.uint8, device=dev)
    rc = lib.pto_attention_pre_quant_launch(descs, 19, ctypes.byref(p), ctypes.c_void_p(ws.data_ptr()), n,
                                            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream), 1)  # sync = 1: returns after the stream has drained
    assert rc == 0, lib.pto_last_error().decode()
    got = {k: v.cpu() for k, v in out.items()}
    got["x_int8"] = ws[:t * h].view(torch.int8).reshape(t, h).cpu()
    return got


def close(a, b, name, half, outliers=1e-3, min_equal=0.98):
    """a against b, [rows, heads * 128] each.  Inside the reference's tolerance except for `outliers` of the elements,
    and every element within 3 x the same tolerance taken on the magnitude of what it was computed from: for a rotary
    dim that is the norm of its (i, i + half) pair, which the rotation preserves - one bf16 step of either input moves a
    result that the rotation has cancelled to near zero by far more than 2^-7 of that result."""
    a, b = a.float(), b.float()
    assert a.shape == b.shape
    assert torch.isfinite(a).all(), name
    if a.numel() == 0:
        return
    err = (a - b).abs()
    ratio = err / (1e-4 + 0.0078125 * b.abs())
    mag = b.abs().reshape(b.shape[0], -1, 128).clone()
    pair = torch.sqrt(mag[..., :half] ** 2 + mag[..., half:2 * half] ** 2)
    mag[..., :half] = pair
    mag[..., half:2 * half] = pair
    worst = (err / (1e-4 + 0.0078125 * mag.reshape(b.shape))).max()
    assert (ratio > 1).float().mean() <= outliers and worst <= 3, \
        f"{name}: {int((ratio > 1).sum())} of {a.numel()} outside the tolerance, worst {float(worst):.2f} x"
    assert (a == b).float().mean() >= min_equal, f"{name}: only {(a == b).float().mean():.4f} bit-equal"


def check(case, got):
    gold = op.attention_pre_quant(case)
    assert torch.equal(got["residual_res"], gold["residual_res"])
    diff = (got["x_int8"].int() - gold["x_int8"].int()).abs()
    if diff.numel():
        assert diff.max() <= 1, f"quantised row off by {int(diff.max())}"
        assert (diff == 0).float().mean() >= 0.999, f"{int((diff != 0).sum())} of {diff.numel()} quantised values differ"
    tail = op.heads_from_x_int8(case, got["x_int8"])
    assert torch.equal(got["value"], tail["value"]), "value from the product's quantised row"
    half = case["cos"].shape[-1]
    close(got["key"], tail["key"], "key from the product's quantised row", half)
    close(got["query"], tail["query"], "query from the product's quantised row", half)
    same = (diff == 0).all(dim=1)
    assert torch.equal(got["value"][same], gold["value"][same]), "value end to end"
    for name in ("key", "query"):
        close(got[name][same], gold[name][same], name + " end to end", half)


@pytest.fixture(scope="module")
def cuda():
    assert torch.cuda.is_available()
    return torch.device("cuda:0")


def test_reference_shape(cuda):
    """8 tokens, hidden 5120, 12 + 1 + 1 heads of 128, rotary on 64 dims (glm_attention_pre_quant.py:510-519)."""
    case = op.make_case(8, seed=11)
    got = run(case, cuda)
    check(case, got)
    via_operator = run_operator(case, cuda)
    for name in ("query", "key", "value", "residual_res"):
        assert torch.equal(via_operator[name], got[name])


def test_reference_test_distribution(cuda):
    """The reference test's inputs, all uniform in [0, 1) (:536-555): most of the quantised row saturates at 1."""
    case = op.make_case(8, realistic=False, seed=12)
    check(case, run(case, cuda))


@pytest.mark.parametrize("t", [1, 5, 11, 33, 64, 100])
def test_token_counts(cuda, t):
    """The reference's dynamic batch sizes (:527-532: 8, 5, 11, 2) and counts around the 32-token tile of the kernel."""
    case = op.make_case(t, h=1024, q_heads=4, kv_heads=2, seed=20 + t)
    check(case, run(case, cuda))


@pytest.mark.parametrize("t,h,q_heads,kv_heads", [(128, 1024, 4, 2), (200, 5120, 12, 1), (300, 6400, 30, 3), (513, 256, 2, 1)])
def test_prefill_token_counts(cuda, t, h, q_heads, kv_heads):
    """Prefill sizes over all projection kernels: token counts that end inside a tile, a contraction split into several
    workgroups with a short last split (6400 = 50 stages of 128), a contraction of two stages taken whole."""
    case = op.make_case(t, h=h, q_heads=q_heads, kv_heads=kv_heads, seed=t + h)
    check(case, run(case, cuda))


def test_whole_model_heads(cuda):
    """All 96 query and 8 key / value heads of GLM-4.5 on one device."""
    case = op.make_case(16, q_heads=96, kv_heads=8, seed=13)
    check(case, run(case, cuda))


@pytest.mark.parametrize("t,q_heads,kv_heads,half", [(128, 3, 1, 20), (129, 2, 1, 64), (1300, 48, 2, 32), (1500, 48, 2, 8), (1800, 48, 2, 1),
                                                     (2100, 47, 2, 32), (9, 62, 1, 32), (31, 60, 3, 32)])
def test_prefill_in_one_split(cuda, t, q_heads, kv_heads, half):
    """A short contraction, which the tiles of 256 outputs take in one split: their workgroups finish their heads themselves.  Tiles
    of 128, 160, 192, 224 and 256 tokens with a remainder, an odd number of heads, rotary halves of whole and of broken pieces (the
    first two cases run the streamed kernel and 128 x 128 tiles)."""
    case = op.make_case(t, h=256, q_heads=q_heads, kv_heads=kv_heads, half=half, seed=40 + t)
    check(case, run(case, cuda))


@pytest.mark.parametrize("t,h,q_heads,kv_heads,half", [
    (33, 5120, 12, 1, 32), (128, 6400, 14, 1, 20), (128, 1024, 15, 1, 64), (129, 6400, 12, 1, 64), (160, 256, 30, 1, 20), (192, 5120, 12, 2, 1), (160, 5120, 26, 2, 1), (161, 256, 26, 2, 32),
    (193, 512, 3, 1, 20), (200, 256, 2, 1, 64), (257, 1024, 12, 1, 8), (288, 256, 30, 1, 64), (289, 1024, 12, 1, 32), (33, 512, 31, 1, 32)])
def test_projection_kernels_at_the_edges_of_their_ranges(cuda, t, h, q_heads, kv_heads, half):
    """Up to 16 heads: streamed up to 128 tokens, 128 x 128 tiles up to 192 and from 257 to 288; up to 32 heads: 128 x 128 tiles
    from 33 to 160 tokens; wider tiles elsewhere.  Short last splits, token tiles with remainders of 1 to all rows."""
    case = op.make_case(t, h=h, q_heads=q_heads, kv_heads=kv_heads, half=half, seed=t + h + half)
    check(case, run(case, cuda))


@pytest.mark.parametrize("t,q_heads,kv_heads,half,scales", [
    (1300, 48, 2, 16, "plain"), (1500, 48, 2, 32, "least"), (1800, 48, 2, 16, "signs"), (2100, 47, 2, 32, "zeros"), (1025, 47, 2, 16, "below"),
    (1300, 48, 2, 32, "most"), (1301, 48, 2, 64, "below"), (1499, 48, 2, 8, "above")])
def test_heads_finished_on_the_tiles_have_the_bits_of_the_head_kernel(cuda, t, q_heads, kv_heads, half, scales):
    """Tiles in one split against the streamed kernel with its head kernel, bit by bit, on the first and the last tokens and around the
    tiles' borders: pairs of rotary dims inside a wave's tile (16 and 32 a half) and across, scales at both ends of the range in
    which a quotient is taken by the reciprocal (2^-60 to 2^60), beyond it, negative and zero."""
    case = op.make_case(t, h=256, q_heads=q_heads, kv_heads=kv_heads, half=half, seed=70 + t)
    deq = case["atten_qkv_deq_scale"]
    n = deq.numel()
    if scales == "signs":
        deq[torch.arange(n) % 5 == 0] *= -1
    elif scales == "zeros":
        deq[torch.arange(n) % 3 == 0] = 0
        deq[:128] = 0
    elif scales != "plain":
        deq[torch.arange(n) % 7 == 0] = {"least": 2.0 ** -60, "below": 2.0 ** -75, "most": 2.0 ** 60, "above": 2.0 ** 61}[scales]
    full = run(case, cuda)
    rows = ("hidden_states", "residual", "cos", "sin")
    for t0 in (0, 124, 188, 252, t - 8):
        got = run({k: v[t0:t0 + 8].contiguous() if k in rows else v for k, v in case.items()}, cuda)
        for name in ("query", "key", "value"):
            assert torch.isfinite(got[name]).all()
            assert torch.equal(got[name], full[name][t0:t0 + 8]), (t0, name)


def test_a_tokens_bits_do_not_depend_on_the_projection_kernel(cuda):
    # int32 sums are exact and the head epilogues the same operations: streamed, 128 x 128 and wide tiles in one and in several splits
    case = op.make_case(300, h=1024, seed=3)
    rows = ("hidden_states", "residual", "cos", "sin")
    full = run(case, cuda)
    for t in (20, 33, 128, 150, 200, 256, 260):
        got = run({k: v[:t].contiguous() if k in rows else v for k, v in case.items()}, cuda)
        for name in ("query", "key", "value", "residual_res"):
            assert torch.equal(got[name], full[name][:t]), (t, name)


@pytest.mark.parametrize("h,half", [(256, 64), (6144, 16), (6400, 1), (16384, 32)])
def test_hidden_sizes_and_rotary_widths(cuda, h, half):
    """The narrowest and the widest hidden size, both sides of the switch between the two norm kernels, full and
    minimal rotary width."""
    case = op.make_case(7, h=h, q_heads=2, kv_heads=1, half=half, seed=h + half)
    check(case, run(case, cuda))


@pytest.mark.parametrize("t,q_heads,kv_heads", [(8, 30, 3), (40, 60, 6)])
def test_several_stages_per_workgroup_with_a_short_last_split(cuda, t, q_heads, kv_heads):
    """Shapes with enough workgroups for the projection kernel to take two (first case) or four (second) stages of 256
    contraction rows per workgroup; hidden 6400 = 25 stages leaves the last split with a single one."""
    case = op.make_case(t, h=6400, q_heads=q_heads, kv_heads=kv_heads, seed=t + q_heads)
    check(case, run(case, cuda))


@pytest.mark.parametrize("t,h,q_heads,kv_heads", [(1, 256, 2, 1), (1, 5120, 12, 1), (2, 6144, 12, 1), (3, 5120, 24, 2), (4, 512, 3, 1), (4, 5120, 96, 8),
                                                  (3, 1280, 94, 9), (2, 5888, 176, 2), (1, 6144, 150, 2), (4, 6144, 150, 2), (5, 5120, 12, 1), (4, 6400, 2, 1)])
def test_norm_in_the_projection(cuda, t, h, q_heads, kv_heads):
    """Up to 4 tokens and hidden 6144 the norm is the projection's workgroups' own: one, two and four stages to a workgroup with and without
    a short last one, one to four tokens; in place of the residual (a kernel of its own there), the same bits."""
    case = op.make_case(t, h=h, q_heads=q_heads, kv_heads=kv_heads, seed=t + h)
    got = run(case, cuda)
    check(case, got)
    from pypto_amd.glm_v4_5 import glm_attention_pre_quant as impl
    for place in ("hidden_states", "residual"):
        on = {k: case[k].to(cuda) for k in NAMES}
        out = outputs(case, cuda)
        impl.attention_pre_quant(*[on[k] for k in NAMES], out["query"], out["key"], out["value"], on[place])
        for name in ("query", "key", "value"):
            assert torch.equal(out[name].cpu(), got[name]), (place, name)
        assert torch.equal(on[place].cpu(), got["residual_res"]), place


@pytest.mark.parametrize("t,h,q_heads", [(5, 2304, 2), (6, 2048, 2), (7, 4096, 3), (9, 4352, 12), (160, 6144, 12), (161, 5120, 2), (33, 5888, 24)])
def test_norm_by_pieces(cuda, t, h, q_heads):
    """5 to 160 tokens of hidden 2304 to 6144: a row's pieces on two and three workgroups, the last one short and whole; in place of an input
    a workgroup has the row, the same bits."""
    case = op.make_case(t, h=h, q_heads=q_heads, kv_heads=1, seed=t + h)
    got = run(case, cuda)
    check(case, got)
    from pypto_amd.glm_v4_5 import glm_attention_pre_quant as impl
    for place in ("hidden_states", "residual"):
        on = {k: case[k].to(cuda) for k in NAMES}
        out = outputs(case, cuda)
        impl.attention_pre_quant(*[on[k] for k in NAMES], out["query"], out["key"], out["value"], on[place])
        for name in ("query", "key", "value"):
            assert torch.equal(out[name].cpu(), got[name]), (place, name)
        assert torch.equal(on[place].cpu(), got["residual_res"]), place


@pytest.mark.parametrize("t,h,q_heads", [(1, 5120, 2), (4, 2048, 12), (3, 6144, 96), (6, 5120, 2), (9, 2304, 12)])
def test_norms_of_infinities_and_nan(cuda, t, h, q_heads):
    """Rows with an infinity, with infinities that cancel, a NaN, and the largest finite values, whose squares overflow: the norm in the
    projection and the norm by pieces give the bits of the workgroup per row, which has them where the sums take an input's place."""
    case = op.make_case(t, h=h, q_heads=q_heads, kv_heads=1, seed=t + h)
    x, r, inf = case["hidden_states"], case["residual"], float("inf")
    x[0, 5] = inf
    if t > 1:
        x[1, h - 1], r[1, h - 1] = inf, -inf
        r[1, 70] = torch.finfo(torch.bfloat16).max
    if t > 2:
        r[2, 1] = float("nan")
    if t > 3:
        x[3, ::7] = torch.finfo(torch.bfloat16).max
    got = run(case, cuda)
    from pypto_amd.glm_v4_5 import glm_attention_pre_quant as impl
    on = {k: case[k].to(cuda) for k in NAMES}
    out = outputs(case, cuda)
    impl.attention_pre_quant(*[on[k] for k in NAMES], out["query"], out["key"], out["value"], on["residual"])
    for name in ("query", "key", "value"):
        assert torch.equal(out[name].cpu().view(torch.int16), got[name].view(torch.int16)), name
    a, b = on["residual"].cpu(), got["residual_res"]
    assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(0.0), b.nan_to_num(0.0))
    assert not torch.isfinite(b[0]).all()


@pytest.mark.parametrize("h", [256, 1024, 1280, 2560, 2816, 4096, 4352, 5120, 5376, 8192, 8448, 12544])
def test_partial_sums_of_any_number_of_splits(cuda, h):
    """1, 4, 5, 10, 11, 16, 17, 20, 21, 32, 33 and 49 splits of the contraction: up to one group of loads and more, whole and with a rest."""
    case = op.make_case(6, h=h, q_heads=2, kv_heads=1, seed=h)
    check(case, run(case, cuda))


def test_saturation_at_both_ends(cuda):
    """A quantisation scale of 1000: nine in ten values of the quantised row are clamped at -128 or 127."""
    case = op.make_case(4, h=4096, q_heads=2, kv_heads=1, seed=14)
    case["atten_qkv_input_scale_reciprocal"] = torch.full((4096,), 1000.0).to(torch.bfloat16)
    gold = op.attention_pre_quant(case)
    x = gold["x_int8"].int()
    assert (x == 127).float().mean() > 0.4 and (x == -128).float().mean() > 0.4
    check(case, run(case, cuda))


def test_sums_beyond_fp32_integers(cuda):
    """A large offset puts the whole quantised row at 127 and the weights are 126 or 127: int32 sums of about 2^26, which
    the conversion to fp32 rounds (to multiples of 4) before the dequantisation scale."""
    case = op.make_case(4, h=4096, q_heads=2, kv_heads=1, seed=17)
    case["atten_qkv_input_offset"] = torch.full((4096,), 30000.0).to(torch.bfloat16)
    case["atten_qkv_weight"] = torch.where(case["atten_qkv_weight"] >= 0, 127, 126).to(torch.int8)
    gold = op.attention_pre_quant(case)
    assert (gold["x_int8"] == 127).all()
    acc = gold["x_int8"].int() @ case["atten_qkv_weight"].int()
    assert acc.min() > 2 ** 25 and (acc % 4 != 0).any()
    check(case, run(case, cuda))


def test_empty(cuda):
    case = op.make_case(0, h=512, q_heads=2, kv_heads=1)
    got = run_operator(case, cuda)
    assert got["query"].shape == (0, 256)
    check(case, run(case, cuda))


def test_outputs_feed_the_paged_attention(cuda):
    """The operator's query / key / value as the newest rows of the GQA decode attention's inputs: the chain agrees with
    the oracle chain (attention golden: oracle/gqa.py)."""
    from oracle import gqa
    from pypto_amd.glm_v4_5 import glm_attention
    b, nq, nkv, d, bs = 4, 12, 1, 128, 128
    case = op.make_case(b, seed=15)
    got = run_operator(case, cuda)
    gold = op.attention_pre_quant(case)
    g = torch.Generator().manual_seed(16)
    act = torch.tensor([5, 130, 256, 77], dtype=torch.int32)
    blocks = 12
    table = torch.arange(blocks, dtype=torch.int32)[torch.randperm(blocks, generator=g)].reshape(b, 3)
    kc = torch.randn(blocks, bs, nkv, d, generator=g).to(torch.bfloat16)
    vc = torch.randn(blocks, bs, nkv, d, generator=g).to(torch.bfloat16)

    def scatter(kc, vc, src):
        kc, vc = kc.clone(), vc.clone()
        for i in range(b):
            pos = int(act[i]) - 1
            kc[table[i, pos // bs], pos % bs] = src["key"][i].reshape(nkv, d)
            vc[table[i, pos // bs], pos % bs] = src["value"][i].reshape(nkv, d)
        return kc, vc

    kg, vg = scatter(kc, vc, got)
    ko, vo = scatter(kc, vc, gold)
    want = gqa.attention_flash(gold["query"].reshape(b, nq, d), ko, vo, table, act, d ** -0.5)
    out = torch.zeros(b, nq, d, dtype=torch.bfloat16, device=cuda)
    glm_attention.attention(got["query"].reshape(b, nq, d).to(cuda), kg.to(cuda), vg.to(cuda), table.to(cuda),
                            act.to(cuda), out, d ** -0.5)
    torch.cuda.synchronize()
    a, w = out.cpu().float(), want.float()
    assert ((a - w).abs() <= 1e-2 + 2e-2 * w.abs()).all()


def test_errors(cuda):
    from pypto_amd.error import FeError
    case = op.make_case(2, h=512, q_heads=2, kv_heads=1, seed=1)
    bad = dict(case, atten_qkv_quant_bias=case["atten_qkv_quant_bias"].float())
    with pytest.raises(AssertionError):
        run_operator(bad, cuda)
    bad = dict(case, atten_qkv_deq_scale=case["atten_qkv_deq_scale"][:-1].contiguous())
    with pytest.raises(FeError, match="entries"):
        run_operator(bad, cuda)
    bad = dict(case, hidden_states=case["hidden_states"][:, :500].contiguous(), residual=case["residual"][:, :500].contiguous())
    with pytest.raises(FeError):
        run_operator(bad, cuda)
