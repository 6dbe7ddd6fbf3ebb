"""GPU parity: fused MLA prolog + lightning-indexer prolog (HIP, through the C ABI).

Two bars.  (1) Plumbing: the fused call must give what the two operators give when called one after the other with the
MLA prolog's q_norm / q_norm_scale handed over by the caller - bit for bit for every MLA output and for the indexer's
query (integer GEMM, same epilogue); the indexer's key path and weights sum x @ [w_k | w_proj] in a different order when
fused (the product rides along in the MLA prolog's first kernel), so there: int8 within 1, fp16 within one bf16 step.
(2) Against the oracle's composition of
the two goldens: the MLA outputs as in test_gpu_mla_prolog; the indexer outputs inherit the (rare, one-step) q_norm
differences of the MLA stage, which is why the reference widens q_int8's tolerance to 2 here
(deepseekv32_mla_indexer_prolog_quant.py:824): int8 within 2 everywhere and equal in at least 95 % of the places, scales
and weights within one bf16 step.
"""
import pytest
import torch

from oracle import mla_prolog as op
from test_gpu_indexer_prolog import WEIGHTS_REL, weights_allowance
from test_gpu_mla_prolog import FEW, check_rope_cache

pytestmark = pytest.mark.gpu
EPS = 1e-5


def _impl():
    from pypto_amd.deepseek_v32_exp import lightning_indexer_prolog_quant_impl as ip
    from pypto_amd.deepseek_v32_exp import mla_indexer_prolog_quant_impl as fused
    from pypto_amd.deepseek_v32_exp import mla_prolog_quant_impl as mla
    return mla, ip, fused


def _buffers(mla_case, idx_case, dev):
    t, r = mla_case["x"].shape[0], mla_case["w_dq"].shape[1]
    n, ni = mla_case["w_uk"].shape[0], idx_case["w_proj"].shape[1]
    m = {k: v.to(dev) for k, v in mla_case.items()}
    i = {k: v.to(dev) for k, v in idx_case.items()}
    z = lambda shape, dt: torch.zeros(shape, dtype=dt, device=dev)  # noqa: E731
    out = {"q_norm": z((t, r), torch.int8), "q_norm_scale": z((t, 1), torch.float32),
           "q_nope": z((t, n, 512), torch.bfloat16), "q_rope": z((t, n, 64), torch.bfloat16),
           "kv_cache": m["kv_cache"].clone(), "kr_cache": m["kr_cache"].clone(), "k_scale_cache": m["k_scale_cache"].clone(),
           "q_int8": z((t, ni, 128), torch.int8), "q_scale": z((t, ni, 1), torch.float16),
           "k_cache": i["k_cache"].clone(), "idx_k_scale_cache": i["k_scale_cache"].clone(),
           "weights": z((t, ni), torch.float16)}
    return m, i, out


def run_fused(mla_case, idx_case, dev, entry="mla_indexer_prolog_quant_d"):
    mla, ip, fused = _impl()
    m, i, o = _buffers(mla_case, idx_case, dev)
    getattr(fused, entry)(
        m["x"], m["w_dq"], m["w_uq_qr"], m["w_qb_scale"], m["w_uk"], m["w_dkv_kr"], m["gamma_cq"], m["gamma_ckv"], m["cos"],
        m["sin"], m["cache_index"], o["kv_cache"], o["kr_cache"], o["k_scale_cache"], i["w_qb"], i["w_qb_scale"], i["w_k"],
        i["w_proj"], i["ln_gamma"], i["ln_beta"], i["hadamard_q"], i["hadamard_k"], o["k_cache"], o["idx_k_scale_cache"],
        o["q_nope"], o["q_rope"], o["kv_cache"], o["kr_cache"], o["k_scale_cache"], o["q_int8"], o["q_scale"], o["k_cache"],
        o["idx_k_scale_cache"], o["weights"], EPS, EPS, "PA_BSND", mla.MlaTileConfig(), ip.IndexerPrologQuantAttr(eps=1e-6),
        ip.IndexerPrologQuantConfigs(), mla.RopeTileShapeConfig([32, 64], [32, 32, 128], [16, 128, 128, 128]))
    torch.cuda.synchronize()
    return {k: v.cpu() for k, v in o.items() if k not in ("q_norm", "q_norm_scale")}


def run_separate(mla_case, idx_case, dev):
    mla, ip, _ = _impl()
    m, i, o = _buffers(mla_case, idx_case, dev)
    mla.mla_prolog_quant_d(
        m["x"], m["w_dq"], m["w_uq_qr"], m["w_qb_scale"], m["w_uk"], m["w_dkv_kr"], m["gamma_cq"], m["gamma_ckv"], m["cos"],
        m["sin"], m["cache_index"], o["kv_cache"], o["kr_cache"], o["k_scale_cache"], o["q_norm"], o["q_norm_scale"],
        o["q_nope"], o["q_rope"], o["kv_cache"], o["kr_cache"], o["k_scale_cache"], EPS, EPS, "PA_BSND", mla.MlaTileConfig(),
        mla.RopeTileShapeConfig([32, 64], [32, 32, 128], [16, 128, 128, 128]))
    ip.lightning_indexer_prolog_quant(
        m["x"], o["q_norm"], o["q_norm_scale"], i["w_qb"], i["w_qb_scale"], i["w_k"], i["w_proj"], i["ln_gamma"],
        i["ln_beta"], m["cos"], m["sin"], i["hadamard_q"], i["hadamard_k"], o["k_cache"], o["idx_k_scale_cache"],
        m["cache_index"], o["q_int8"], o["q_scale"], o["k_cache"], o["idx_k_scale_cache"], o["weights"],
        ip.IndexerPrologQuantConfigs(), ip.IndexerPrologQuantAttr(eps=1e-6))
    torch.cuda.synchronize()
    return {k: v.cpu() for k, v in o.items()}


def check_against_oracle(mla_case, idx_case, got):
    gm, gi = op.mla_indexer_prolog(mla_case, idx_case, EPS, EPS, 1e-6)
    rows = mla_case["cache_index"]

    def ints(a, b, name, tol, min_equal):
        diff = (a.int() - b.int()).abs()
        # (a quantisation scale that moved by one bf16 step of the row's largest value moves a quantised value v by
        # v / 128 steps: in the upper half of the int8 range that is one more step than the value's own rounding)
        assert (diff <= tol + (b.int().abs() >= 64).int()).all(), f"{name}: off by {int(diff.max())}"
        assert (diff == 0).float().mean() >= min_equal, f"{name}: {(diff != 0).float().mean():.4f} of the values differ"

    def close(a, b, name, rel=2.0 ** -7, atol=1e-8, outliers=0.0):
        a, b = a.float().flatten(), b.float().flatten()
        assert torch.isfinite(a).all(), name
        ratio = (a - b).abs() / (rel * b.abs() + atol)
        assert int((ratio > 1).sum()) <= (max(outliers * ratio.numel(), FEW) if outliers else 0) and ratio.max() <= 3, \
            f"{name}: {int((ratio > 1).sum())} values out of tolerance, worst {float(ratio.max())} x"

    ints(got["kv_cache"].view(-1, 512)[rows], gm["kv_cache"].view(-1, 512)[rows], "kv_cache", 1, 0.98)
    close(got["k_scale_cache"].view(-1, 4)[rows], gm["k_scale_cache"].view(-1, 4)[rows], "k_scale_cache", rel=2.0 ** -6)  # see test_gpu_mla_prolog
    close(got["q_nope"], gm["q_nope"], "q_nope", 0.0078125, 0.005, outliers=5e-3)   # see test_gpu_mla_prolog
    close(got["q_rope"], gm["q_rope"], "q_rope", 0.0078125, 0.005, outliers=5e-3)
    check_rope_cache(mla_case, got["kr_cache"], gm["kr_cache"], EPS)   # see test_gpu_mla_prolog
    # (the reference's widened tolerance of 2; with a q_lora_rank of 128 a flipped q_norm value is one of only 128 terms
    # of a product and moves it by more: 3 there)
    ints(got["q_int8"], gi["q_int8"], "q_int8", 2 if mla_case["w_dq"].shape[1] >= 256 else 3, 0.95)
    # (the golden's index queries come from the golden's q_norm, the product's from its own: a q_norm value that rounded
    # the other way shifts the 128 values of a head a little, on top of the one bf16 step their own rounding can move,
    # which is why q_int8 gets 2 above; a query scale follows the largest of them, so two bf16 steps here.  The tight
    # check of this stage is that the fused call gives the bits of the separate calls, whose index prolog is tested
    # against the oracle from one and the same q_norm.)
    close(got["q_scale"], gi["q_scale"], "q_scale", rel=2.0 ** -6)
    ints(got["k_cache"].view(-1, 128)[rows], gi["k_cache"].view(-1, 128)[rows], "idx k_int8", 1, 0.98)
    close(got["idx_k_scale_cache"].view(-1)[rows], gi["k_scale_cache"].view(-1)[rows], "idx k_scale")
    close(got["weights"], gi["weights"], "weights", rel=WEIGHTS_REL, atol=weights_allowance(idx_case).flatten())


def same_as_separate(fused, sep, idx_case):
    for k, v in fused.items():
        if k in ("k_cache", "idx_k_scale_cache", "weights"):
            continue
        assert torch.equal(v, sep[k]), f"{k}: fused and separate calls differ"
    assert (fused["k_cache"].int() - sep["k_cache"].int()).abs().max() <= 1
    assert (fused["k_cache"] == sep["k_cache"]).float().mean() >= 0.999
    a, b = fused["idx_k_scale_cache"].float(), sep["idx_k_scale_cache"].float()
    assert ((a - b).abs() <= 2.0 ** -7 * b.abs() + 1e-8).all(), "idx_k_scale_cache"
    # weights near zero are sums that cancel: there the summation order shows at the fp32 level of the h terms
    a, b = fused["weights"].float(), sep["weights"].float()
    assert ((a - b).abs() <= WEIGHTS_REL * b.abs() + weights_allowance(idx_case)).all(), "weights"


def test_reference_case_b4_s2_fused_equals_separate_and_oracle(cuda):
    # the reference's enabled test test_b_4_s1_2_tilebs_8_d: b=4, two new tokens per sequence, model sizes
    mla_case, idx_case = op.make_fused_case(4, 2, 1024, seed=21)
    fused = run_fused(mla_case, idx_case, cuda)
    sep = run_separate(mla_case, idx_case, cuda)
    same_as_separate(fused, sep, idx_case)
    check_against_oracle(mla_case, idx_case, fused)


def test_prefill_entry_ragged_tiles_small_sizes(cuda):
    mla_case, idx_case = op.make_fused_case(37, 1, 300, seed=22, n_idx=64, h=512, q_lora_rank=256, n=4)
    fused = run_fused(mla_case, idx_case, cuda, entry="mla_indexer_prolog_quant_p")
    sep = run_separate(mla_case, idx_case, cuda)
    same_as_separate(fused, sep, idx_case)
    check_against_oracle(mla_case, idx_case, fused)


def test_prefill_sizes_fused_equals_separate_and_oracle(cuda):
    # 128 tokens and more: the first product of both calls runs the kernel that owns an output tile, and so does the
    # separate call's int8 product (exact, so still the fused call's bits)
    # (the two int8 products of the fused call always share a launch; above 128 tokens that of the wide tiles)
    for b, seed in ((150, 24), (300, 25)):
        mla_case, idx_case = op.make_fused_case(b, 1, 300, seed=seed, n_idx=64, h=1280, q_lora_rank=256, n=4)
        fused = run_fused(mla_case, idx_case, cuda, entry="mla_indexer_prolog_quant_p")
        sep = run_separate(mla_case, idx_case, cuda)
        same_as_separate(fused, sep, idx_case)
        check_against_oracle(mla_case, idx_case, fused)


@pytest.mark.parametrize("t,n,r,h", [(1100, 2, 128, 512), (1290, 4, 256, 256), (1540, 2, 128, 256), (300, 6, 384, 2304)])
def test_prefill_index_query_tiles(cuda, t, n, r, h):
    """Index query tiles of 160, 192, 224 and 128 tokens: the product is exact and the rest the same operations, so the bits of
    the separate call's 128-token tiles; the last also a contraction of three splits, the latent rank no multiple of 256."""
    mla_case, idx_case = op.make_fused_case(t, 1, 64, seed=50 + n, n_idx=64, h=h, q_lora_rank=r, n=n)
    fused = run_fused(mla_case, idx_case, cuda, entry="mla_indexer_prolog_quant_p")
    same_as_separate(fused, run_separate(mla_case, idx_case, cuda), idx_case)
    check_against_oracle(mla_case, idx_case, fused)


@pytest.mark.parametrize("t,n", [(128, 6), (129, 6), (160, 64), (193, 2), (256, 2)])
def test_products_around_the_narrow_tiles_limit(cuda, t, n):
    # up to 128 tokens tiles of 128 outputs, above of 256 with a remainder of one token, half a tile (two heads) and whole tiles
    mla_case, idx_case = op.make_fused_case(t, 1, 64, seed=80 + n, n_idx=64, h=256, q_lora_rank=128, n=n)
    fused = run_fused(mla_case, idx_case, cuda, entry="mla_indexer_prolog_quant_p")
    same_as_separate(fused, run_separate(mla_case, idx_case, cuda), idx_case)
    check_against_oracle(mla_case, idx_case, fused)


@pytest.mark.parametrize("t,n", [(33, 6), (64, 6), (65, 2), (96, 128), (97, 6), (128, 258), (129, 128), (160, 96), (161, 96), (150, 64), (145, 72), (145, 74)])
def test_streamed_products_of_33_to_160_tokens(cuda, t, n):
    # token blocks of 32: two to five with remainders of one and all rows, the last head count of one round of workgroups and one past
    # it (258 heads), and the tiles that take over
    mla_case, idx_case = op.make_fused_case(t, 1, 64, seed=90 + n, n_idx=64, h=512, q_lora_rank=384, n=n)
    fused = run_fused(mla_case, idx_case, cuda, entry="mla_indexer_prolog_quant_p")
    same_as_separate(fused, run_separate(mla_case, idx_case, cuda), idx_case)
    check_against_oracle(mla_case, idx_case, fused)


@pytest.mark.parametrize("t,n", [(257, 64), (775, 64), (1447, 16), (1762, 8), (961, 64), (1793, 64)])
def test_index_head_tiles_ahead_of_the_query_tiles(cuda, t, n):
    # one launch holds the index heads' tiles of all token tiles (32 each), then the query product's (48, 12 or 6 each): three to
    # twelve token tiles of 128, 160 (three shapes), 192 and 224 tokens, the last of 135, 7, 2 tokens or one
    mla_case, idx_case = op.make_fused_case(t, 1, 64, seed=80 + n, n_idx=64, h=256, q_lora_rank=128, n=n)
    fused = run_fused(mla_case, idx_case, cuda, entry="mla_indexer_prolog_quant_p")
    same_as_separate(fused, run_separate(mla_case, idx_case, cuda), idx_case)
    check_against_oracle(mla_case, idx_case, fused)


@pytest.mark.parametrize("t,n,r", [(673, 64, 256), (768, 64, 128), (1793, 38, 384)])
def test_index_head_tiles_of_256_tokens(cuda, t, n, r):
    # tiles of 256 tokens, whose halves of 128 go through LDS one after the other: the last tile of 161 tokens (both halves), of all
    # 256 and of one (the second half empty)
    mla_case, idx_case = op.make_fused_case(t, 1, 64, seed=100 + n, n_idx=64, h=256, q_lora_rank=r, n=n)
    fused = run_fused(mla_case, idx_case, cuda, entry="mla_indexer_prolog_quant_p")
    same_as_separate(fused, run_separate(mla_case, idx_case, cuda), idx_case)
    check_against_oracle(mla_case, idx_case, fused)


@pytest.mark.parametrize("t,n,h", [(300, 6, 1280), (300, 2, 2816)])
def test_x_product_in_splits_of_whole_stages(cuda, t, n, h):
    # two splits of ten stages of 64 rows, and of 15, 15 and 14: no multiples of the 256 that the hidden size is one of
    mla_case, idx_case = op.make_fused_case(t, 1, 64, seed=110 + n, n_idx=64, h=h, q_lora_rank=128, n=n)
    fused = run_fused(mla_case, idx_case, cuda, entry="mla_indexer_prolog_quant_p")
    same_as_separate(fused, run_separate(mla_case, idx_case, cuda), idx_case)
    check_against_oracle(mla_case, idx_case, fused)


@pytest.mark.parametrize("t,n,r", [(1, 2, 128), (32, 16, 384), (31, 66, 256), (5, 128, 1536), (9, 130, 128)])
def test_absorbed_product_behind_the_query_product(cuda, t, n, r):
    # beside the index heads', to 128 heads (130: kernels of their own).  The separate call of up to 64 heads is two kernels: the same bits
    mla_case, idx_case = op.make_fused_case(t, 1, 300, seed=150 + n, n_idx=64, h=512, q_lora_rank=r, n=n)
    fused = run_fused(mla_case, idx_case, cuda)
    same_as_separate(fused, run_separate(mla_case, idx_case, cuda), idx_case)
    check_against_oracle(mla_case, idx_case, fused)


@pytest.mark.parametrize("t,n,r", [(33, 4, 128), (64, 128, 256), (97, 66, 128), (129, 80, 384), (160, 128, 256), (160, 66, 256), (257, 60, 384),
                                   (300, 128, 1536), (330, 130, 128), (410, 128, 128), (512, 128, 256), (1030, 128, 128)])
def test_absorbed_product_behind_tiles(cuda, t, n, r):
    # all tokens beside 128 outputs, blocks of 32 tokens with the last ones missing; tiles of 128 to 256 tokens, one and two rounds of
    # workgroups and more, where the units go out in turn; 66 and 130 heads end with half a unit of rotary dims and begin rounds of the XCDs anew.
    # Separate calls of few heads are two kernels: the same bits
    mla_case, idx_case = op.make_fused_case(t, 1, 300, seed=160 + n, n_idx=64, h=512, q_lora_rank=r, n=n)
    fused = run_fused(mla_case, idx_case, cuda)
    same_as_separate(fused, run_separate(mla_case, idx_case, cuda), idx_case)
    check_against_oracle(mla_case, idx_case, fused)


@pytest.mark.parametrize("t,n_idx,r,h", [(257, 128, 1664, 256), (258, 64, 1536, 2304), (259, 64, 384, 1280), (1284, 128, 128, 512), (261, 64, 128, 5120), (300, 128, 1664, 8192), (270, 64, 256, 9216)])
def test_norms_by_wavefronts(cuda, t, n_idx, r, h):
    # above 256 tokens and with at most eight splits of x's product (nine: a workgroup to a chain), four tokens to a workgroup: one, two and three
    # of them and all in the last; one, two, three, five and eight splits; latent ranks past 1536 and no multiple of 256; two index heads to a lane.  The MLA outputs are the
    # bits of the separate call, whose norms are workgroups of their own
    mla_case, idx_case = op.make_fused_case(t, 1, 64, seed=130 + n_idx, n_idx=n_idx, h=h, q_lora_rank=r, n=2)
    fused = run_fused(mla_case, idx_case, cuda, entry="mla_indexer_prolog_quant_p")
    same_as_separate(fused, run_separate(mla_case, idx_case, cuda), idx_case)
    check_against_oracle(mla_case, idx_case, fused)


def test_norms_by_wavefronts_of_infinities_and_nan(cuda):
    # tokens whose sums are infinite, not a number, and overflow when squared: what the workgroups' norms of the separate call make of them
    mla_case, idx_case = op.make_fused_case(258, 1, 64, seed=135, n_idx=64, h=2304, q_lora_rank=384, n=2)
    x = mla_case["x"]
    x[0, 5], x[1, 7], x[2] = float("inf"), float("nan"), torch.finfo(torch.bfloat16).max / 4
    x[257, 9] = -float("inf")
    idx_case["x"] = x
    fused, sep = run_fused(mla_case, idx_case, cuda, entry="mla_indexer_prolog_quant_p"), run_separate(mla_case, idx_case, cuda)
    for k in ("q_nope", "q_rope", "kv_cache", "kr_cache", "k_scale_cache", "q_int8", "q_scale"):
        a, b = fused[k].float(), sep[k].float()
        assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(0.0), b.nan_to_num(0.0)), k
    assert fused["q_nope"][3:257].isfinite().all() and not fused["kr_cache"].isfinite().all()


def test_query_weights_whose_last_rows_lie_beyond_4_gb(cuda):
    # 33 tokens, 128 rows of 33818880 outputs: the last heads' results are the bits of a call of these heads alone
    n, r = 176140, 128
    mla_case, idx_case = op.make_fused_case(33, 1, 64, seed=121, n_idx=64, h=256, q_lora_rank=r, n=2)
    small = run_fused(mla_case, idx_case, cuda)
    g = torch.Generator(device=cuda).manual_seed(122)
    many = dict(mla_case, w_uq_qr=torch.randint(-127, 128, (r, n * 192), generator=g, device=cuda, dtype=torch.int8),
                w_qb_scale=torch.full((n * 192, 1), 1e-3, device=cuda), w_uk=torch.zeros((n, 128, 512), dtype=torch.bfloat16, device=cuda))
    many["w_uq_qr"][:, -384:], many["w_qb_scale"][-384:], many["w_uk"][-2:] = (mla_case[k].to(cuda) for k in ("w_uq_qr", "w_qb_scale", "w_uk"))
    big = run_fused(many, idx_case, cuda)
    assert torch.equal(big["q_nope"][:, -2:], small["q_nope"]) and torch.equal(big["q_rope"][:, -2:], small["q_rope"])


def test_index_head_counts_without_the_side_by_side_kernels(cuda):
    # 32 index heads: x @ w_proj is half an output tile wide, so the fused entry runs the two operators back to back
    mla_case, idx_case = op.make_fused_case(5, 1, 300, seed=23, n_idx=32, h=512, q_lora_rank=256, n=4)
    fused = run_fused(mla_case, idx_case, cuda)
    sep = run_separate(mla_case, idx_case, cuda)
    for k, v in fused.items():
        assert torch.equal(v, sep[k]), f"{k}: fused and separate calls differ"


def test_decode_layer_front_end_chain(cuda):
    """One decode layer's attention front end as three chained calls on the GPU, each stage checked against the oracle
    on the previous stage's actual outputs: fused prolog -> (indexer query, weights, updated index cache) -> lightning
    indexer -> top-k rows -> sparse flash attention over the updated int8 MLA cache with the prolog's query."""
    from _cases import run_indexer, run_sfa
    from test_gpu_indexer import check_topk
    from test_gpu_sfa import full_check
    b, s1, s2 = 2, 2, 3000
    mla_case, idx_case = op.make_fused_case(b, s1, s2, seed=25)
    got = run_fused(mla_case, idx_case, cuda)
    n_pages = got["k_cache"].shape[0]
    ci = {"query": got["q_int8"], "q_scale": got["q_scale"].reshape(b * s1, 64), "weights": got["weights"],
          "key_cache": got["k_cache"], "k_scale": got["idx_k_scale_cache"].reshape(n_pages, 128, 1),
          "act_seq": [s2] * b, "block_table": mla_case["block_table"], "b": b, "s1": s1, "selected_count": 2048,
          "block_size": 128}
    topk = run_indexer(ci, cuda)
    check_topk(ci, topk)
    ca = {"b": b, "s1": s1, "nq": 128, "topk": 2048, "block_size": 128, "softmax_scale": 192 ** -0.5, "act_seq": [s2] * b,
          "q": torch.cat([got["q_nope"], got["q_rope"]], dim=-1).reshape(b, s1, 128, 576),
          "kn": got["kv_cache"].view(-1, 512), "kr": got["kr_cache"].view(-1, 64),
          "kn_scales": got["k_scale_cache"].view(-1, 4), "topk_indices": topk.reshape(b * s1, 2048),
          "block_table": mla_case["block_table"]}
    # the newest token of a query's causal range is its own, just-written cache row: it must be reachable
    new_rows = mla_case["cache_index"].reshape(b, s1)
    assert (ca["kn_scales"][new_rows.reshape(-1)] > 0).all()
    full_check(run_sfa(ca, cuda), ca, "prolog -> indexer -> attention")


def test_no_tokens_is_a_no_op(cuda):
    """An empty batch (t = 0) is accepted by all three prolog entries and touches nothing."""
    mla_case, idx_case = op.make_fused_case(2, 1, 256, seed=24, n_idx=64, h=512, q_lora_rank=256, n=4)
    for k in ("x", "cos", "sin", "cache_index"):
        mla_case[k] = mla_case[k][:0].contiguous()
    idx_case.update(x=mla_case["x"], cos=mla_case["cos"], sin=mla_case["sin"], k_cache_index=mla_case["cache_index"])
    fused = run_fused(mla_case, idx_case, cuda)
    sep = run_separate(mla_case, idx_case, cuda)
    for got in (fused, sep):
        assert torch.equal(got["kv_cache"], mla_case["kv_cache"]) and torch.equal(got["kr_cache"], mla_case["kr_cache"])
        assert torch.equal(got["k_scale_cache"], mla_case["k_scale_cache"])
        assert torch.equal(got["k_cache"], idx_case["k_cache"])
        assert torch.equal(got["idx_k_scale_cache"], idx_case["k_scale_cache"])
        assert got["q_nope"].shape == (0, 4, 512) and got["q_int8"].shape == (0, 64, 128)


def test_errors(cuda):
    from pypto_amd.error import FeError
    mla_case, idx_case = op.make_fused_case(2, 1, 256, seed=1, n_idx=32, h=512, q_lora_rank=256, n=4)
    with pytest.raises(FeError, match="heads"):
        run_fused(mla_case, dict(idx_case, w_proj=idx_case["w_proj"][:, :16].contiguous()), cuda)
    with pytest.raises(FeError, match="int64|INT64"):
        run_fused(dict(mla_case, cache_index=mla_case["cache_index"].int()), idx_case, cuda)
