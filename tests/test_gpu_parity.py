"""Parity of the HIP path (through the C ABI) with the CPU oracle and with the
reference's own outputs (golden fixtures).  All tests need an MI355X."""
from __future__ import annotations

import os

import pytest
import torch

from conftest import load_golden
from helpers import (KEEP_TIE_TOL, tune, SELECT_SCORE_TOL, assert_keep_matches, assert_keep_within_exact_bound, build_inputs,
                     device_exact_gate, device_objects, exact_gate, oracle_raw, record_swaps, score_tolerance,
                     selection_score_tol)
from oracle import compaction as ocp
from oracle import scoring as osc
from oracle import selection as osel
from triattention_amd import ops, synth

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def small(**kw):
    base = dict(name="t", num_layers=2, num_q_heads=8, num_kv_heads=2, head_dim=128, seq_lens=(300,),
                budget=96, block_size=16, window_size=12, rope_theta=1e6, index=7)
    base.update(kw)
    return synth.Workload(**base)


def run_scores(w, inp, aggregation="mean", round_start=None, **flags):
    caches, kv, batch, sc = device_objects(w, inp, DEV, round_start=round_start, aggregation=aggregation, **flags)
    raw, ws = ops.score_paged(kv, batch, sc)
    torch.cuda.synchronize()
    return raw.cpu(), (caches, kv, batch, sc, ws)


SCORE_CASES = {
    "c0": dict(w=synth.config(0)),
    "gqa4_two_layers": dict(w=small()),
    "ragged_batch": dict(w=small(seq_lens=(300, 17, 1000, 256, 513), num_layers=3)),
    "hkv8": dict(w=small(num_q_heads=32, num_kv_heads=8, seq_lens=(700, 90))),
    "hkv4_g7": dict(w=small(num_q_heads=28, num_kv_heads=4, seq_lens=(333,))),
    "g8": dict(w=small(num_q_heads=64, num_kv_heads=8, seq_lens=(260,))),
    "g1": dict(w=small(num_q_heads=2, num_kv_heads=2, seq_lens=(129,))),
    "hkv1": dict(w=small(num_q_heads=4, num_kv_heads=1, seq_lens=(200,))),
    "hkv16": dict(w=small(num_q_heads=16, num_kv_heads=16, seq_lens=(150,))),
    "d64": dict(w=small(head_dim=64, num_q_heads=16, num_kv_heads=8, seq_lens=(270,))),
    "d256": dict(w=small(head_dim=256, seq_lens=(140,))),
    "interleaved": dict(w=small(rope_style="interleaved")),
    "fp16": dict(w=small(kv_dtype="fp16")),
    "fp16_interleaved_ragged": dict(w=small(kv_dtype="fp16", rope_style="interleaved", seq_lens=(300, 17, 1000, 513),
                                            num_layers=3)),
    "fp16_g8": dict(w=small(kv_dtype="fp16", num_q_heads=16, num_kv_heads=2, seq_lens=(700, 90))),
    "block32": dict(w=small(block_size=32, seq_lens=(500, 31))),
    "block_not_pow2": dict(w=small(block_size=24, seq_lens=(301,))),
    "kv_axis1": dict(w=small(seq_lens=(290, 64)), kv_axis=1),
    "llama3": dict(w=small(rope_theta=5e5, rope_scaling="llama3")),
    "max_agg": dict(w=small(seq_lens=(300, 40)), aggregation="max"),
    "max_agg_d64": dict(w=small(head_dim=64, seq_lens=(100,)), aggregation="max"),
    # max aggregation on the matrix cores (bf16 keys, head dimension 128)
    "max_agg_interleaved_ragged": dict(w=small(rope_style="interleaved", seq_lens=(1300, 17, 513, 1), num_layers=3),
                                       aggregation="max"),
    "max_agg_g8": dict(w=small(num_q_heads=16, num_kv_heads=2, seq_lens=(700, 90)), aggregation="max"),
    "max_agg_hkv4_g7": dict(w=small(num_q_heads=28, num_kv_heads=4, seq_lens=(333,)), aggregation="max"),
    "max_agg_g1_hkv3": dict(w=small(num_q_heads=3, num_kv_heads=3, seq_lens=(129, 600)), aggregation="max"),
    "max_agg_block_not_pow2": dict(w=small(block_size=24, seq_lens=(301, 1025)), aggregation="max"),
    "max_agg_kv_axis1_block32": dict(w=small(block_size=32, seq_lens=(290, 64)), kv_axis=1, aggregation="max"),
    "max_agg_fp16": dict(w=small(kv_dtype="fp16", seq_lens=(200,)), aggregation="max"),
    "no_mlr": dict(w=small(), disable_mlr=True),
    "no_trig": dict(w=small(), disable_trig=True),
    "no_trig_max": dict(w=small(), disable_trig=True, aggregation="max"),
    "late_round": dict(w=small(), round_start=[70000]),
    # fp8 e4m3 keys with per-(token, head) scales: no reference counterpart, oracle = dequantise then score
    "fp8": dict(w=small(kv_dtype="fp8", seq_lens=(300, 45))),
    "fp8_hkv8_llama3": dict(w=small(kv_dtype="fp8", num_q_heads=32, num_kv_heads=8, rope_theta=5e5,
                                    rope_scaling="llama3", seq_lens=(530,))),
    "fp8_interleaved": dict(w=small(kv_dtype="fp8", rope_style="interleaved")),
    "fp8_d64": dict(w=small(kv_dtype="fp8", head_dim=64, num_q_heads=16, num_kv_heads=8, seq_lens=(270,))),
    "fp8_d256_hkv2": dict(w=small(kv_dtype="fp8", head_dim=256, num_q_heads=4, num_kv_heads=2, seq_lens=(140,))),
    "fp8_block24": dict(w=small(kv_dtype="fp8", block_size=24, seq_lens=(301,))),
    "fp8_max_agg": dict(w=small(kv_dtype="fp8", seq_lens=(200,)), aggregation="max"),
}


@pytest.mark.parametrize("name", list(SCORE_CASES))
def test_raw_scores_match_oracle(name):
    case = dict(SCORE_CASES[name])
    w = case.pop("w")
    kv_axis = case.pop("kv_axis", 0)
    agg = case.pop("aggregation", "mean")
    rs = case.pop("round_start", None)
    inp = build_inputs(w, kv_axis)
    print(f"case={name} workload={w}", flush=True)
    raw, _ = run_scores(w, inp, agg, rs, **case)
    for b, t in enumerate(w.seq_lens):
        rstart = rs[b] if rs is not None else t
        want = oracle_raw(w, inp, b, rstart, agg, **case)
        for l in range(w.num_layers):
            got = raw[b, l, :t].transpose(0, 1)                  # [A, T]
            err = (got - want[l]).abs()
            tol = score_tolerance(want[l])                        # 1e-3 relative to per-head RMS
            assert bool((err <= tol).all()), (name, b, l, float(err.max()), float(tol.min()))


@pytest.mark.parametrize("name", ["max_agg", "max_agg_interleaved_ragged", "max_agg_g8", "max_agg_hkv4_g7",
                                  "max_agg_block_not_pow2"])
def test_max_aggregation_on_matrix_cores_matches_the_vector_unit_kernel(name, monkeypatch):
    """Keys are exact in bf16 and the coefficients enter in three bf16 pieces, so the matrix-core
    kernel agrees with the vector-unit kernel to fp32 rounding (1e-5 of the per-head RMS, a
    hundred times tighter than the bound against the oracle); the per-tile sums behind the
    statistics are compared through the selection scores."""
    case = dict(SCORE_CASES[name])
    w = case.pop("w")
    kv_axis = case.pop("kv_axis", 0)
    inp = build_inputs(w, kv_axis)
    print(f"case={name} workload={w}", flush=True)
    out = {}
    for kernel in ("mfma", "valu"):
        tune(max_kernel=kernel)
        caches, kv, batch, sc = device_objects(w, inp, DEV, aggregation="max")
        raw, ws = ops.score_paged(kv, batch, sc)
        sel = ops.SelectConfig(window_size=w.window_size)
        keep, fin = ops.select(kv, batch, sc, sel, raw, ws, want_scores=True)
        torch.cuda.synchronize()
        out[kernel] = (raw.clone(), fin.clone())
    h = w.num_kv_heads
    for b, t in enumerate(w.seq_lens):
        got, want = out["mfma"][0][b, :, :t], out["valu"][0][b, :, :t]          # [L, T, A]
        rms = want.pow(2).mean(dim=1, keepdim=True).sqrt().clamp_min(1e-30)
        assert float(((got - want).abs() / rms).max()) <= 1e-5, (name, b)
        fm, fv = out["mfma"][1][b * h:(b + 1) * h, :t], out["valu"][1][b * h:(b + 1) * h, :t]
        finite = torch.isfinite(fv)
        assert torch.equal(torch.isfinite(fm), finite)
        if bool(finite.any()):
            assert float((fm[finite] - fv[finite]).abs().max()) <= SELECT_SCORE_TOL * float(fv[finite].abs().max()), (name, b)


@pytest.mark.parametrize("seed", range(int(os.environ.get("TRIATTN_TEST_RANDOM_SHAPES", "32")) // 2))
def test_max_aggregation_on_matrix_cores_on_random_shapes(seed, monkeypatch):
    """Seeded random head layouts, ragged lengths, block sizes, RoPE pairings and cache layouts: the
    matrix-core max-aggregation scorer against the vector-unit kernel."""
    import random
    r = random.Random(5000 + seed)
    hkv, g = r.choice([1, 2, 3, 4, 8]), r.choice([1, 2, 3, 4, 5, 7, 8])
    seq_lens = tuple(r.choice([1, 15, 16, 17, 97, 130, 511, 513, 700, 1100]) for _ in range(r.choice([1, 2, 3])))
    w = small(num_q_heads=hkv * g, num_kv_heads=hkv, seq_lens=seq_lens, num_layers=r.choice([1, 2, 3]),
              block_size=r.choice([8, 16, 24, 32]), rope_style=r.choice(["half", "interleaved"]), index=500 + seed)
    SCORE_CASES[f"random_max{seed}"] = dict(w=w, kv_axis=r.choice([0, 1]), aggregation="max")
    try:
        test_max_aggregation_on_matrix_cores_matches_the_vector_unit_kernel(f"random_max{seed}", monkeypatch)
    finally:
        del SCORE_CASES[f"random_max{seed}"]


def test_head_major_output_layout():
    w = small(seq_lens=(200, 77))
    inp = build_inputs(w)
    caches, kv, batch, sc = device_objects(w, inp, DEV)
    a, ws = ops.score_paged(kv, batch, sc)
    b, _ = ops.score_paged(kv, batch, sc, ws, head_major=True)
    torch.cuda.synchronize()
    for i, t in enumerate(w.seq_lens):
        assert torch.equal(a[i, :, :t].transpose(1, 2), b[i, :, :, :t])


def test_dense_keys_entry():
    """[B, H, T, D] keys without a block table (core/scoring.py:79-204 call shape)."""
    g = torch.Generator().manual_seed(3)
    b, h, t, d = 2, 4, 150, 128
    keys = torch.randn(b, h, t, d, generator=g).to(torch.bfloat16)
    qc = torch.randn(1, h, d // 2, 2, generator=g)
    qa = qc.pow(2).sum(-1).sqrt() + torch.rand(1, h, d // 2, generator=g)
    fs = 0.5 + torch.rand(1, h, d // 2, generator=g)
    omega = synth.rope_inv_freq(small())
    offs = synth.geometric_offsets()
    kd = keys.to(DEV)
    kv = ops.PagedKV.from_dense_keys(kd)
    batch = ops.StepBatch(DEV, [t, t], round_start=[500, 500])
    sc = ops.ScoreConfig(ops.fold_stats(qc.to(DEV), qa.to(DEV), fs.to(DEV)), omega.to(DEV), offs.to(DEV))
    raw, _ = ops.score_paged(kv, batch, sc, head_major=True)
    torch.cuda.synchronize()
    want = osc.raw_scores(keys, qc[0], qa[0], omega, offs, fs[0], 500)
    got = raw[:, 0].cpu()
    assert bool(((got - want).abs() <= score_tolerance(want)).all())


SELECT_CASES = {
    "default": dict(w=small(seq_lens=(300, 1000, 97))),
    "c0": dict(w=synth.config(0)),
    "prefill": dict(w=small(seq_lens=(400, 222)), prefill=[30, 5], protect_prefill=True),
    "nonorm": dict(w=small(seq_lens=(300,)), normalize=False),
    "layer_max": dict(w=small(seq_lens=(300,), num_layers=3), layer_reduce="max"),
    "under_budget": dict(w=small(seq_lens=(50, 96, 97))),
    "no_window": dict(w=small(seq_lens=(300,), window_size=0)),
    "hkv8": dict(w=small(num_q_heads=32, num_kv_heads=8, seq_lens=(700,), budget=256)),
    "g7": dict(w=small(num_q_heads=28, num_kv_heads=4, seq_lens=(333,))),
}


@pytest.mark.parametrize("name", list(SELECT_CASES))
def test_group_selection_matches_oracle(name):
    case = dict(SELECT_CASES[name])
    w = case.pop("w")
    prefill = case.pop("prefill", None)
    protect = case.pop("protect_prefill", False)
    normalize = case.pop("normalize", True)
    layer_reduce = case.pop("layer_reduce", "mean")
    inp = build_inputs(w)
    print(f"case={name} workload={w}", flush=True)
    caches, kv, batch, sc = device_objects(w, inp, DEV, prefill_lens=prefill)
    raw, ws = ops.score_paged(kv, batch, sc)
    sel = ops.SelectConfig(normalize=normalize, window_size=w.window_size, protect_prefill=protect,
                           layer_reduce=layer_reduce)
    keep, fin = ops.select(kv, batch, sc, sel, raw, ws, want_scores=True)
    torch.cuda.synchronize()
    keep, fin = keep.cpu(), fin.cpu()
    h = w.num_kv_heads
    total_swapped = compared = 0
    for b, t in enumerate(w.seq_lens):
        k = min(w.budget, t)
        oraw = oracle_raw(w, inp, b, t)
        okw = dict(normalize=normalize, window_size=w.window_size, prefill_len=prefill[b] if prefill else 0,
                   protect_prefill=protect, chunk_tokens=osel.score_chunk_tokens(w.block_size, t), layer_agg=layer_reduce)
        want, ofin = osel.group_keep_per_head(oraw, h, w.budget, **okw)
        got = keep[b * h:(b + 1) * h, :k].long()
        assert bool((got[:, 1:] > got[:, :-1]).all())            # strictly ascending
        if ofin is None:
            assert torch.equal(got, want)
            continue
        dfin = fin[b * h:(b + 1) * h, :t]
        finite = torch.isfinite(ofin)
        assert torch.equal(torch.isfinite(dfin), finite)
        if not bool(finite.any()):        # every token guarded: any k of them is as good as another
            continue
        scale = ofin[finite].abs().max()
        assert float((dfin[finite] - ofin[finite]).abs().max()) <= selection_score_tol(oraw) * float(scale)
        # An index may differ from the oracle's only where the exact score is no further from the exact
        # threshold than the oracle's own fp32 evaluation is from the exact one on these very inputs.
        fin64, bound = exact_gate(oraw, h, **okw)
        total_swapped += assert_keep_within_exact_bound(got, want, fin64, k, bound)
        compared += h * k
    record_swaps(f"two_pass_vs_oracle:{name}", total_swapped, compared)
    if not name.startswith("random"):
        assert total_swapped == 0, (name, total_swapped)


@pytest.mark.parametrize("seed", range(int(os.environ.get("TRIATTN_TEST_RANDOM_SHAPES", "32")) // 2))
def test_group_selection_matches_oracle_on_random_shapes(seed):
    """Seeded random head layouts, key types, head dimensions, lengths and guards: scores and kept
    sets of the two-pass kernels against the oracle."""
    import random
    r = random.Random(2000 + seed)
    hkv, g = r.choice([1, 2, 3, 4, 8]), r.choice([1, 2, 4, 7, 8])
    seq_lens = tuple(r.choice([1, 17, 64, 97, 130, 300, 513, 700]) for _ in range(r.choice([1, 2, 3])))
    w = small(kv_dtype=r.choice(["bf16", "bf16", "fp16", "fp8"]), head_dim=r.choice([64, 128, 128, 256]),
              num_q_heads=hkv * g, num_kv_heads=hkv, seq_lens=seq_lens, num_layers=r.choice([1, 2, 3]),
              budget=r.choice([16, 96, 200]), block_size=r.choice([8, 16, 32]), window_size=r.choice([0, 12, 40]),
              rope_style=r.choice(["half", "interleaved"]), index=300 + seed)
    case = dict(w=w, normalize=r.random() < 0.8, layer_reduce=r.choice(["mean", "mean", "max"]))
    if r.random() < 0.3:
        case.update(prefill=[r.randrange(0, t + 1) for t in seq_lens], protect_prefill=True)
    SELECT_CASES[f"random{seed}"] = case
    try:
        test_group_selection_matches_oracle(f"random{seed}")
    finally:
        del SELECT_CASES[f"random{seed}"]


@pytest.mark.parametrize("tag,kw", [
    ("default", dict()),
    ("chunk64_prefill", dict(protect_prefill=True)),
    ("nonorm", dict(normalize=False)),
    ("aggmax", dict(aggregation="max")),
])
@pytest.mark.parametrize("path", ["two_pass", "resident_mfma", "resident_valu"])
@pytest.mark.parametrize("fixture", ["selector_group.pt", "selector_group_d128.pt"])
def test_group_selection_matches_reference_golden(tag, kw, path, fixture, monkeypatch):
    """Keep sets written by the reference's own selector (paged group branch), through the
    two-pass path and through both resident kernels."""
    if path != "two_pass":
        tune(resident_kernel=path.split("_")[1])
    gold = load_golden(fixture)
    layers, hkv, t, d = gold["keys"].shape
    hq = gold["q_mean_complex"].shape[1]
    bs, pool = int(gold["block_size"]), int(gold["pool_blocks"])
    ids = gold["block_ids"].tolist()
    caches = []
    for l in range(layers):
        kvc = torch.zeros(2, pool, bs, hkv, d, dtype=torch.bfloat16)
        tok = torch.arange(t)
        blk = torch.tensor(ids)[tok // bs]
        kvc[0, blk, tok % bs] = gold["keys"][l].transpose(0, 1)
        kvc[1, blk, tok % bs] = gold["values"][l].transpose(0, 1)
        caches.append(kvc.to(DEV))
    kv = ops.PagedKV.from_kv_caches(caches)
    budget = int(gold["budget"])
    batch = ops.StepBatch(DEV, [t], round_start=[int(gold["round_start"])], budgets=budget,
                          block_tables=[ids], prefill_lens=[int(gold["prefill_len"])])
    folded = ops.fold_stats(gold["q_mean_complex"].to(DEV), gold["q_abs_mean"].to(DEV),
                            torch.ones(layers, hq, d // 2, device=DEV))
    sc = ops.ScoreConfig(folded, gold["omega"].to(DEV), synth.geometric_offsets(device=DEV),
                         kw.get("aggregation", "mean"))
    sel = ops.SelectConfig(normalize=kw.get("normalize", True), window_size=int(gold["window"]),
                           protect_prefill=kw.get("protect_prefill", False))
    if path == "two_pass":
        raw, ws = ops.score_paged(kv, batch, sc)
        keep, _ = ops.select(kv, batch, sc, sel, raw, ws)
    else:
        if ops.select_path(kv, batch, sc, sel) != path:
            pytest.skip(f"this setting runs {ops.select_path(kv, batch, sc, sel)}")
        keep, _, ws = ops.select_paged(kv, batch, sc, sel)
        assert ws.status() == 0
    torch.cuda.synchronize()
    want = gold[f"group_{tag}_keep"]
    got = keep.cpu().long()
    diff = sum(len(set(got[h].tolist()) ^ set(want[h].tolist())) for h in range(hkv))
    assert diff == 0, f"{diff} indices differ from the reference's keep set"
    assert torch.equal(got, want)


@pytest.mark.parametrize("tag,protect", [("default", False), ("chunk64_prefill", True)])
@pytest.mark.parametrize("fixture,path,copies,workgroups", [
    ("selector_c1_shape.pt", "two_pass", 1, None),
    ("selector_c1_shape.pt", "resident_mfma", 1, 5),    # five tiles of 1024 tokens on the eight-wave instance the benchmark times
    ("selector_c1_shape.pt", "resident_mfma", 3, 15),   # three requests in one launch, each must come out as the single one
    ("selector_c1_shape.pt", "resident_mfma", 3, 10),   # ... and in two launches (two sequences, then one)
    ("selector_c1_shape.pt", "resident_valu", 1, 5),
    # eight query heads per KV head (Qwen3-32B attention), 37 % kept: tiles of 512 tokens on the instance the
    # 8 x 32768-token configuration runs (two groups of query heads)
    ("selector_c2_shape.pt", "two_pass", 1, None),
    ("selector_c2_shape.pt", "resident_mfma", 1, 10),
    ("selector_c2_shape.pt", "resident_mfma", 2, 10),   # two requests, one launch each
    # head dimension 64 with the statistics shipped for GPT-OSS-120B and its YaRN frequencies
    ("selector_gpt_oss_shape.pt", "two_pass", 1, None),
    ("selector_gpt_oss_shape.pt", "resident_mfma", 1, 10),
    ("selector_gpt_oss_shape.pt", "resident_mfma", 2, 20),
])
def test_group_selection_at_the_benchmarked_head_shape_matches_reference_golden(tag, protect, fixture, path, copies,
                                                                                workgroups, monkeypatch):
    """The reference's keep sets for a 5000-token request of 32 query / 8 KV heads of 128 (budget
    2048, window 128; written by tests/golden/make_c1_shape_golden.py): its variance streams over
    two 4096-token chunks and its chunked top-k merges.  The resident matrix-core kernel is
    pinned to the instance and tile size of the 16 x 16384-token benchmark step (tiles of 1024
    tokens, workgroups of eight waves) by pretending the device holds only five workgroups.
    Gate: the reference's rows, except indices whose double-precision selection score lies no
    further from the double-precision threshold than the reference's own fp32 selection scores lie
    from the double-precision ones on this fixture (helpers.exact_gate)."""
    from golden.hashed_inputs import checksum, hashed_rows
    gold = load_golden(fixture)
    layers, hq, hkv, d, t, bs = (int(x) for x in gold["shape"])
    keys = hashed_rows(int(gold["key_seed"]), layers, hkv, t, d)
    assert checksum(keys) == int(gold["key_checksum"]), "the hashed keys differ from the ones the golden was written for"
    pool = int(gold["pool_blocks"])
    ids = gold["block_ids"]
    tok = torch.arange(t)
    caches = []
    for l in range(layers):
        kvc = torch.zeros(2, pool * copies, bs, hkv, d, dtype=torch.bfloat16)
        for c in range(copies):
            kvc[0, ids[tok // bs] + c * pool, tok % bs] = keys[l].transpose(0, 1)
        caches.append(kvc.to(DEV))
    tables = [(ids + c * pool).tolist() for c in range(copies)]
    if path != "two_pass":
        tune(resident_kernel=path.split("_")[1])
        tune(resident_workgroups=workgroups)
    kv = ops.PagedKV.from_kv_caches(caches)
    budget = int(gold["budget"])
    batch = ops.StepBatch(DEV, [t] * copies, round_start=[int(gold["round_start"])] * copies, budgets=budget,
                          block_tables=tables, prefill_lens=[int(gold["prefill_len"])] * copies)
    folded = ops.fold_stats(gold["q_mean_complex"].to(DEV), gold["q_abs_mean"].to(DEV),
                            torch.ones(layers, hq, d // 2, device=DEV))
    sc = ops.ScoreConfig(folded, gold["omega"].to(DEV), synth.geometric_offsets(device=DEV))
    sel = ops.SelectConfig(window_size=int(gold["window"]), protect_prefill=protect,
                           allow_resident=path != "two_pass")
    assert ops.select_path(kv, batch, sc, sel) == path
    keep, _, ws = ops.select_paged(kv, batch, sc, sel)
    assert ws.status() == 0
    want = gold[f"group_{tag}_keep"].long()
    okeep, ofin, fin64, bound = _head_shape_oracle(fixture, tag)
    # The oracle reproduces the reference's keep set: exactly on the machine the golden was written on
    # (tests/test_oracle_selection.py asserts that); torch's CPU reductions associate differently on other
    # CPUs, so here the two may differ where the fp32 evaluation itself is undecided.
    assert_keep_within_exact_bound(okeep, want, fin64, int(gold["budget"]), bound)
    scale = float(ofin[torch.isfinite(ofin)].abs().max())
    # (the reference's own distance from exact arithmetic: 8e-6 of the largest score with one 4096-token
    # chunk, 2e-5 with chunks of 64; the kernels, which sum the statistics in double, sit 6e-6 .. 7e-6 away)
    assert 0 < bound <= 5e-5 * scale
    got = keep.cpu().long().view(copies, hkv, budget)
    swapped = 0
    for c in range(copies):
        # Identical to the reference's rows except where the reference's own fp32 rounding, not the
        # formula, decides on which side of the threshold an index falls.
        swapped += assert_keep_within_exact_bound(got[c], want, fin64, budget, bound)
    record_swaps(f"reference_golden_{fixture[9:-9]}_shape:{path}:{copies}x:{workgroups}:{tag}", swapped,
                 copies * hkv * budget)
    assert swapped <= 2 * copies, swapped


_HEAD_SHAPE_ORACLE: dict = {}


def _head_shape_oracle(fixture, tag):
    """Keep rows, fp32 and double-precision selection scores of the CPU oracle for a head-shape golden."""
    if (fixture, tag) not in _HEAD_SHAPE_ORACLE:
        from golden.hashed_inputs import hashed_rows
        gold = load_golden(fixture)
        layers, hq, hkv, d, t, bs = (int(x) for x in gold["shape"])
        keys = hashed_rows(int(gold["key_seed"]), layers, hkv, t, d)
        offs = osc.geometric_offsets(65536)
        raw = [osc.raw_scores(keys[l].float().repeat_interleave(hq // hkv, dim=0), gold["q_mean_complex"][l],
                              gold["q_abs_mean"][l], gold["omega"], offs, torch.ones(hq, d // 2), int(gold["round_start"]))
               for l in range(layers)]
        kw = dict(chunk_tokens=64, protect_prefill=True) if tag == "chunk64_prefill" else dict(chunk_tokens=4096)
        kw.update(window_size=int(gold["window"]), prefill_len=int(gold["prefill_len"]))
        _HEAD_SHAPE_ORACLE[(fixture, tag)] = osel.group_keep_per_head(raw, hkv, int(gold["budget"]), **kw) + exact_gate(raw, hkv, **kw)
    return _HEAD_SHAPE_ORACLE[(fixture, tag)]


@pytest.mark.parametrize("fixture", ["selector_group.pt", "selector_group_d128.pt"])
@pytest.mark.parametrize("tag,kw", [("default", dict()), ("nonorm", dict(normalize=False))])
def test_layer_selection_matches_reference_golden(tag, kw, fixture):
    """Per-layer selection (runtime/selector_hf.py:473-677) against the reference's output for layer 1."""
    gold = load_golden(fixture)
    layers, hkv, t, d = gold["keys"].shape
    hq = gold["q_mean_complex"].shape[1]
    bs, pool = int(gold["block_size"]), int(gold["pool_blocks"])
    ids = gold["block_ids"].tolist()
    caches = []
    for l in range(layers):
        kvc = torch.zeros(2, pool, bs, hkv, d, dtype=torch.bfloat16)
        tok = torch.arange(t)
        blk = torch.tensor(ids)[tok // bs]
        kvc[0, blk, tok % bs] = gold["keys"][l].transpose(0, 1)
        caches.append(kvc.to(DEV))
    kv = ops.PagedKV.from_kv_caches(caches)
    batch = ops.StepBatch(DEV, [t], round_start=[int(gold["round_start"])], budgets=int(gold["budget"]),
                          block_tables=[ids], prefill_lens=[int(gold["prefill_len"])])
    folded = ops.fold_stats(gold["q_mean_complex"].to(DEV), gold["q_abs_mean"].to(DEV),
                            torch.ones(layers, hq, d // 2, device=DEV))
    sc = ops.ScoreConfig(folded, gold["omega"].to(DEV), synth.geometric_offsets(device=DEV))
    sel = ops.SelectConfig(normalize=kw.get("normalize", True), window_size=int(gold["window"]), layer_reduce=None)
    raw, ws = ops.score_paged(kv, batch, sc)
    keep, _ = ops.select(kv, batch, sc, sel, raw, ws)
    torch.cuda.synchronize()
    got = keep.cpu().long().view(layers, hkv, -1)[1]
    assert torch.equal(got, gold[f"layer1_{tag}_keep"])


@pytest.mark.parametrize("fixture", ["selector_group.pt", "selector_group_d128.pt"])
@pytest.mark.parametrize("tag,kw", [("default", dict()), ("nonorm", dict(normalize=False))])
def test_one_layer_of_a_per_layer_selection_takes_the_resident_kernel(tag, kw, fixture):
    """The reference's per-layer modes call the selector once per layer (runtime/selector_hf.py:473-747
    from the layer loop): a keep set per layer of a one-layer call is the group selection of that layer,
    so the call takes the resident kernel, or the two short launches that take its place for so little, and still gives the
    reference's rows for layer 1."""
    gold = load_golden(fixture)
    layers, hkv, t, d = gold["keys"].shape
    hq = gold["q_mean_complex"].shape[1]
    bs, pool = int(gold["block_size"]), int(gold["pool_blocks"])
    ids = gold["block_ids"].tolist()
    kvc = torch.zeros(2, pool, bs, hkv, d, dtype=torch.bfloat16)
    tok = torch.arange(t)
    blk = torch.tensor(ids)[tok // bs]
    kvc[0, blk, tok % bs] = gold["keys"][1].transpose(0, 1)
    kv = ops.PagedKV.from_kv_caches([kvc.to(DEV)])
    batch = ops.StepBatch(DEV, [t], round_start=[int(gold["round_start"])], budgets=int(gold["budget"]),
                          block_tables=[ids], prefill_lens=[int(gold["prefill_len"])])
    folded = ops.fold_stats(gold["q_mean_complex"][1:2].to(DEV), gold["q_abs_mean"][1:2].to(DEV),
                            torch.ones(1, hq, d // 2, device=DEV))
    sc = ops.ScoreConfig(folded, gold["omega"].to(DEV), synth.geometric_offsets(device=DEV))
    sel = ops.SelectConfig(normalize=kw.get("normalize", True), window_size=int(gold["window"]), layer_reduce=None)
    for kernel, small_launches in (("auto", 1), ("mfma", 0)):
        tune(resident_kernel=kernel)
        sel.allow_resident = True
        assert ops.describe_plan(kv, batch, sc, sel)["small_launches"] == small_launches
        assert ops.select_path(kv, batch, sc, sel) == "resident_mfma"
        keep, fin, ws = ops.select_paged(kv, batch, sc, sel, want_scores=True)
        sel.allow_resident = False
        assert ops.select_path(kv, batch, sc, sel) == "two_pass"
        keep_t, fin_t, _ = ops.select_paged(kv, batch, sc, sel, want_scores=True)
        torch.cuda.synchronize()
        assert ws.status() == 0
        assert torch.equal(keep.cpu().long().view(hkv, -1), gold[f"layer1_{tag}_keep"])
        assert torch.equal(keep_t.cpu().long().view(hkv, -1), gold[f"layer1_{tag}_keep"])
        a, b = fin.cpu().view(hkv, -1)[:, :t], fin_t.cpu().view(hkv, -1)[:, :t]
        m = torch.isfinite(b)
        assert torch.equal(torch.isfinite(a), m)
        assert float((a[m] - b[m]).abs().max()) <= 1e-4 * float(b[m].abs().max())


@pytest.mark.parametrize("width", [3000, 8192, 16384, 20001, 32768, 40000])
def test_topk_rows_by_width(width):
    """Rows up to 4096 / 8192 / 16384 / 32768 elements are selected from registers (four kernel
    instances), longer ones by the streaming kernel; ties keep the lowest index."""
    g = torch.Generator().manual_seed(width)
    x = torch.randn(6, width, generator=g)
    x[1, 100:width // 2] = 0.5
    x[2, :] = -3.0
    x[3, -50:] = float("inf")
    x[4, ::7] = float("-inf")
    x[5] = torch.round(x[5] * 4) / 4              # many small tie classes
    print(f"topk width={width}", flush=True)
    xd = x.to(DEV)
    for k in (1, 130, 2048, width - 1, width):
        got = ops.topk_rows(xd, k).cpu().long()
        assert torch.equal(got[:, :k], osel.topk_ascending(x, k)), k
    lens = [width, 10, 1, width - 3, 777, width // 2 + 1]
    ks = [5, 20, 1, 2048, 0, width // 3]
    got = ops.topk_rows(xd, ks, lens).cpu().long()
    for r, (n, k) in enumerate(zip(lens, ks)):
        kk = min(k, n)
        if kk:
            assert torch.equal(got[r, :kk], osel.topk_ascending(x[r:r + 1, :n], kk)[0])


@pytest.mark.parametrize("width", [1025, 4096, 4097, 16385, 32768])
def test_topk_rows_bin_edges(width):
    """The histogram pass cuts [min, max] of a row's finite scores into 2048 bins; rows where one bin
    holds nearly everything (an outlier far away, a range beyond the largest float, subnormal steps),
    more guarded tokens than the budget, and scores on both sides of zero."""
    g = torch.Generator().manual_seed(width)
    x = torch.randn(8, width, generator=g)
    x[0, 7] = 3.0e38                              # one outlier: the rest shares the lowest bin
    x[1, 3], x[1, 9] = 3.4e38, -3.4e38            # max - min is not a float
    x[2] = torch.randint(0, 1 << 20, (width,), generator=g).float() * 1.4e-45   # subnormal spacing
    x[3] = 1.0 + torch.randint(0, 3, (width,), generator=g).float() * 1.1920929e-07
    x[4, : width // 2] = float("inf")             # more +inf than most budgets below
    x[5, ::2] = float("-inf")
    x[6] = -x[6].abs() * 1e-30
    x[7, : width - 2] = float("-inf")
    xd = x.to(DEV)
    for k in (1, 2, width // 4, width // 2 + 1, width - 1):
        got = ops.topk_rows(xd, k).cpu().long()
        assert torch.equal(got[:, :k], osel.topk_ascending(x, k)), k


@pytest.mark.parametrize("width", [1026, 4096, 8000, 16384, 32768])
def test_topk_rows_cut_again_where_many_scores_share_a_bin(width):
    """Rows in which one of the equal bins holds more than the 128 scores that are ranked: outliers, long tails,
    clusters closer than a bin on both sides of zero, a few values many times over.  One, two and three cuts of the
    keys, and cuts that end because all that is left is equal."""
    g = torch.Generator().manual_seed(width + 1)
    x = torch.randn(9, width, generator=g)
    step = torch.randint(0, 3000, (width,), generator=g).float() * 2.0 ** -23
    x[0, 5] = 1e30
    x[1] = x[1].sign() * (8 * x[1].abs()).exp()
    x[2] = 1.0 + step
    x[2, 9] = 1e6
    x[3, : width // 2] = 1.0 + step[: width // 2]
    x[3, width // 2:] = -1.0 - step[width // 2:]
    x[3, 11] = -1e20
    x[4] = 2.5
    x[4, 0] = 3e38
    x[5] = torch.randint(-1, 2, (width,), generator=g).float()
    x[5, 1], x[5, 2] = 1e35, -1e35
    x[6, ::3] *= 1e-41
    x[6, 1::3] *= 1e30
    x[7] = (30 * x[7]).exp()
    x[8] = torch.randint(0, 1 << 23, (width,), generator=g).int().view(torch.float32)     # subnormal, any spacing
    x[8, 3] = 1.0
    xd = x.to(DEV)
    for k in (1, 2, width // 4, width // 3 + 1, width // 2, width - 1):
        got = ops.topk_rows(xd, k).cpu().long()
        assert torch.equal(got[:, :k], osel.topk_ascending(x, k)), k


def test_topk_rows_ties_and_order():
    g = torch.Generator().manual_seed(1)
    x = torch.randn(5, 3000, generator=g)
    x[1, 100:400] = 0.5                       # a large tie class straddling the threshold
    x[2, :] = 1.0                             # everything ties
    x[3, -50:] = float("inf")
    x[4, ::7] = float("-inf")
    for k in (1, 17, 256, 2999, 3000):
        got = ops.topk_rows(x.to(DEV), k).cpu().long()
        want = osel.topk_ascending(x, k)
        assert torch.equal(got[:, :k], want), k
    lens = [3000, 10, 1, 2048, 777]
    ks = [5, 20, 1, 2048, 0]
    got = ops.topk_rows(x.to(DEV), ks, lens).cpu().long()
    for r, (n, k) in enumerate(zip(lens, ks)):
        kk = min(k, n)
        if kk:
            assert torch.equal(got[r, :kk], osel.topk_ascending(x[r:r + 1, :n], kk)[0])


def _compact_case(w, kv_axis, shared, per_layer, full, budgets=None):
    inp = build_inputs(w, kv_axis)
    caches = [c.to(DEV) for c in inp["caches"]]
    kv = ops.PagedKV.from_kv_caches(caches, kv_axis=kv_axis)
    budgets = list(budgets) if budgets is not None else [w.budget] * w.num_seqs
    batch = ops.StepBatch(DEV, w.seq_lens, budgets=budgets, block_tables=inp["tables"])
    g = torch.Generator().manual_seed(99)
    rows_per = (w.num_layers if per_layer else 1) * (1 if shared else w.num_kv_heads)
    keep = torch.zeros(w.num_seqs * rows_per, batch.max_budget, dtype=torch.int32)
    for b, t in enumerate(w.seq_lens):
        k = min(budgets[b], t)
        for r in range(rows_per):
            keep[b * rows_per + r, :k] = torch.sort(torch.randperm(t, generator=g)[:k]).values.int()
    before = [c.clone() for c in inp["caches"]]
    ops.compact(kv, batch, keep.to(DEV), keep_per_layer=per_layer, shared=shared, full_permutation=full)
    torch.cuda.synchronize()
    for l in range(w.num_layers):
        want = before[l].clone()
        for b, t in enumerate(w.seq_lens):
            k = min(budgets[b], t)
            base = b * rows_per + (l * (1 if shared else w.num_kv_heads) if per_layer else 0)
            if shared:
                ocp.compact_shared(want, inp["tables"][b], w.block_size, keep[base, :k].long(), t,
                                   kv_axis=kv_axis, full_permutation=full)
            else:
                ocp.compact_per_head(want, inp["tables"][b], w.block_size,
                                     keep[base:base + w.num_kv_heads, :k].long(), t,
                                     kv_axis=kv_axis, full_permutation=full)
        got = caches[l].cpu()
        assert torch.equal(got.view(torch.int16), want.view(torch.int16)), (l,)


@pytest.mark.parametrize("kv_axis", [0, 1])
@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("per_layer", [False, True])
@pytest.mark.parametrize("full", [False, True])
def test_compaction_bit_exact(kv_axis, shared, per_layer, full):
    w = small(seq_lens=(300, 97, 40, 1234), num_layers=2, num_q_heads=8, num_kv_heads=4, budget=96)
    print(f"compact kv_axis={kv_axis} shared={shared} per_layer={per_layer} full={full}", flush=True)
    _compact_case(w, kv_axis, shared, per_layer, full)


def test_compaction_large_budget_and_dims():
    _compact_case(small(seq_lens=(5000,), budget=3000, num_kv_heads=8, num_q_heads=8), 0, False, False, False)
    _compact_case(small(seq_lens=(700,), budget=300, head_dim=64, block_size=32), 0, False, False, False)
    _compact_case(small(seq_lens=(700,), budget=300, head_dim=256, block_size=8), 0, True, False, False)


@pytest.mark.parametrize("seed", range(int(os.environ.get("TRIATTN_TEST_RANDOM_SHAPES", "32"))))
def test_compaction_on_random_shapes(seed):
    """Seeded random head counts, head dimensions, block sizes, ragged lengths, budgets per
    sequence (from a single row to all but a few) and modes, bit-exact against the oracle."""
    import random
    r = random.Random(1000 + seed)
    hkv = r.choice([1, 2, 3, 4, 5, 7, 8, 9, 16])
    nseq = r.choice([1, 2, 3, 6])
    seq_lens = tuple(r.choice([1, 2, 15, 16, 17, 100, 257, 1000, 1500, 2176, 4100]) for _ in range(nseq))
    budgets = [max(1, r.choice([1, 7, t // 8, t // 2, t - 1, t - 128, t, t + 5])) for t in seq_lens]
    w = small(seq_lens=seq_lens, num_layers=r.choice([1, 2, 3]), num_q_heads=hkv, num_kv_heads=hkv,
              head_dim=r.choice([64, 128, 128, 256]), block_size=r.choice([1, 8, 16, 16, 24, 32, 128]),
              budget=max(budgets), index=200 + seed)
    kv_axis, shared = r.choice([0, 1]), r.random() < 0.4
    per_layer, full = r.random() < 0.3, r.random() < 0.25
    print(f"compaction seed={seed} workload={w} budgets={budgets} kv_axis={kv_axis} shared={shared} "
          f"per_layer={per_layer} full={full}", flush=True)
    _compact_case(w, kv_axis, shared, per_layer, full, budgets=budgets)


@pytest.mark.parametrize("heads", [3, 5, 6, 7])
def test_shared_compaction_with_token_rows_that_do_not_divide_a_tile(heads):
    """One index list for all heads moves whole token rows; with 3, 5, 6 or 7 heads a row's
    chunk count does not divide the 1024-chunk tile of the ordered pass, so a tile has spare
    chunk slots (they must not write anything of their own)."""
    print(f"shared compaction heads={heads}", flush=True)
    _compact_case(small(seq_lens=(3000, 500), budget=1500, num_kv_heads=heads, num_q_heads=heads), 0, True, False, False)
    _compact_case(small(seq_lens=(1600,), budget=1500, num_kv_heads=heads, num_q_heads=heads), 1, True, True, False)


@pytest.mark.parametrize("shared", [False, True])
def test_compaction_when_few_tokens_are_dropped_and_budgets_differ(shared):
    """The rows that come from beyond the budget are a short suffix of every keep list when a
    step drops few tokens; the copy of that suffix is launched with few workgroups.  Also a
    batch in which one sequence's own budget is far below the largest one, so its suffix is
    longer than the launch was sized for."""
    kw = dict(num_layers=2, num_q_heads=8, num_kv_heads=4)
    print(f"compact few drops shared={shared}", flush=True)
    _compact_case(small(seq_lens=(1128, 1000, 1064), budget=1000, **kw), 0, shared, False, False)
    _compact_case(small(seq_lens=(1100, 1100, 1100), **kw), 0, shared, False, False, budgets=[1000, 500, 37])
    _compact_case(small(seq_lens=(2176,), budget=2048, num_layers=1, num_q_heads=8, num_kv_heads=8), 1, shared, False, False)


@pytest.mark.parametrize("layers,heads,dim,tokens,budget", [
    (1, 8, 128, 4300, 2049),      # 16 chains: two workgroups per row, one slot beyond an address segment
    (1, 8, 64, 2100, 2048),       # 16 chains of 128-byte rows: whole rows
    (8, 8, 128, 700, 513),        # 128 chains: the last with half rows, one slot beyond a tile
    (16, 8, 256, 300, 100),       # 256 chains: the last with the longest tile
    (17, 8, 128, 2300, 2048),     # 272 chains: 32 KB tiles
    (64, 8, 64, 120, 97),         # 1024 chains: the last of those
    (65, 8, 64, 120, 97),         # 1040 chains: workgroups of 512
    (32, 8, 64, 600, 120),        # 512 chains of a sparse list: still one launch
    (33, 8, 64, 600, 120),        # 528 chains of a sparse list: ordered pass and bulk pass
])
@pytest.mark.parametrize("in_place", [0, 1, -1])
def test_compaction_on_both_sides_of_every_launch_rule(layers, heads, dim, tokens, budget, in_place):
    """The launch depends on how many chains (sequence, layer, K or V, head) there are and on how sparse
    the lists are; rows already in place (a prefix of the list: none, one, all but one) are not touched.
    Rows are copies of bytes: exact."""
    fixed = in_place if in_place >= 0 else budget - 1
    print(f"compact rules {layers}x{heads}x{dim} {tokens}->{budget} fixed={fixed}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(5)
    nb = (tokens + 15) // 16
    cache = torch.randint(-2**15, 2**15, (layers, 2, nb, 16, heads, dim), dtype=torch.int16, device=DEV, generator=g)
    kv_cache = cache.view(torch.bfloat16)
    kv = ops.PagedKV([c[0] for c in kv_cache], [c[1] for c in kv_cache])
    table = torch.randperm(nb, generator=g, device=DEV)
    batch = ops.StepBatch(DEV, [tokens], budgets=budget, block_tables=[table.tolist()])
    tail = torch.rand(heads, tokens - fixed - 1, generator=g, device=DEV).topk(budget - fixed, 1).indices.sort(1).values
    keep = torch.cat([torch.arange(fixed, device=DEV).expand(heads, fixed), tail + fixed + 1], 1).int().contiguous()
    want = cache.clone()
    slot = lambda t: (table[t // 16], t % 16)
    head = torch.arange(heads, device=DEV).unsqueeze(1).expand(heads, budget)
    (sb, so), (db, do) = slot(keep.long()), slot(torch.arange(budget, device=DEV).expand(heads, budget))
    want[:, :, db, do, head] = cache[:, :, sb, so, head]
    ops.compact(kv, batch, keep)
    torch.cuda.synchronize()
    assert torch.equal(cache, want)


@pytest.mark.parametrize("dtype,scales,layers,heads,dim,tokens,budget", [
    ("bf16", False, 136, 1, 128, 6200, 2048),    # 272 chains, a third of the context: one launch up to 2048 entries,
    ("bf16", False, 136, 1, 128, 6200, 2049),    # ... two passes beyond
    ("bf16", False, 129, 8, 64, 300, 100),       # 2064 chains of 128-byte rows: two passes,
    ("bf16", False, 129, 8, 64, 300, 150),       # ... one launch from half of the context on
    ("bf16", False, 17, 8, 256, 330, 110),       # 512-byte rows: two passes at a third of the context,
    ("bf16", False, 17, 8, 256, 330, 111),       # ... one launch above
    ("fp8", False, 17, 8, 64, 600, 120),         # 64-byte rows, 272 chains: two passes at a fifth,
    ("fp8", False, 17, 8, 64, 600, 121),         # ... one launch above
    ("fp8", False, 33, 8, 64, 300, 149),         # 528 chains: two passes below half
    ("fp8", True, 12, 8, 128, 300, 100),         # 192 chains beside the scales: one launch,
    ("fp8", True, 13, 8, 128, 300, 209),         # ... 208: two passes below 70 % of the context,
    ("fp8", True, 13, 8, 128, 300, 210),         # ... one launch from there,
    ("fp8", True, 26, 4, 128, 300, 149),         # ... with four heads from half of it
    ("fp8", True, 26, 4, 128, 300, 150),
])
def test_compaction_on_both_sides_of_the_rule_for_one_launch(dtype, scales, layers, heads, dim, tokens, budget):
    """One launch or two passes depends on the chains, the share and the number of rows that stay, the bytes of a row
    and whether a cache's scales move beside them.  Rows and scales are copies: exact."""
    print(f"one launch or two {dtype} scales={scales} {layers}x{heads}x{dim} {tokens}->{budget}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(7)
    nb, size = (tokens + 15) // 16, 1 if dtype == "fp8" else 2
    raw = torch.randint(0, 256, (layers, 2, nb, 16, heads, dim * size), dtype=torch.uint8, device=DEV, generator=g)
    cache = raw.view(torch.float8_e4m3fn if dtype == "fp8" else torch.bfloat16)
    sc = torch.rand(layers, 2, nb * 16, heads, device=DEV, generator=g)
    sides = [[x[i] for x in sc] if scales else None for i in (0, 1)]
    kv = ops.PagedKV([c[0] for c in cache], [c[1] for c in cache], "half", *sides)
    table = torch.randperm(nb, generator=g, device=DEV)
    batch = ops.StepBatch(DEV, [tokens], budgets=budget, block_tables=[table.tolist()])
    keep = torch.rand(heads, tokens, generator=g, device=DEV).topk(budget, 1).indices.sort(1).values.int().contiguous()
    slot = lambda t: (table[t // 16], t % 16)
    head = torch.arange(heads, device=DEV).unsqueeze(1).expand(heads, budget)
    (sb, so), (db, do) = slot(keep.long()), slot(torch.arange(budget, device=DEV).expand(heads, budget))
    want, want_sc = raw.clone(), sc.clone()
    want[:, :, db, do, head] = raw[:, :, sb, so, head]
    if scales:
        want_sc[:, :, db * 16 + do, head] = sc[:, :, sb * 16 + so, head]
    ops.compact(kv, batch, keep)
    torch.cuda.synchronize()
    assert torch.equal(raw, want) and torch.equal(sc, want_sc)


@pytest.mark.parametrize("axis", [0, 1])
def test_compaction_matches_reference_golden(axis):
    """Full-permutation output written by the reference's compact_request_kv_in_place(_per_head)."""
    g = load_golden("compaction.pt")[f"axis{axis}"]
    bs, t = int(g["block_size"]), int(g["total_tokens"])
    for mode, keep_key, after_key in (("per_head", "keep_per_head", "kv_after_per_head"),
                                      ("shared", "keep_shared", "kv_after_shared")):
        # head_dim 16 is below the kernels' 64: widen rows by viewing 4 tokens... not
        # possible in place, so this fixture is replayed with head_dim padded to 64.
        before = g["kv_before"]
        pad = torch.zeros(*before.shape[:-1], 64, dtype=before.dtype)
        pad[..., :16] = before
        cache = pad.to(DEV)
        kv = ops.PagedKV.from_kv_caches([cache], kv_axis=axis)
        keep = g[keep_key].int()
        keep = keep if keep.ndim == 2 else keep.unsqueeze(0)
        batch = ops.StepBatch(DEV, [t], budgets=int(keep.shape[1]), block_tables=[g["block_ids"].tolist()])
        ops.compact(kv, batch, keep.contiguous().to(DEV), shared=(mode == "shared"), full_permutation=True)
        torch.cuda.synchronize()
        got = cache.cpu()[..., :16]
        assert torch.equal(got.view(torch.int16), g[after_key].view(torch.int16)), mode


def test_compress_step_equals_chained_calls():
    w = small(seq_lens=(300, 1000, 97, 50), num_layers=3, num_q_heads=16, num_kv_heads=4)
    inp = build_inputs(w)
    caches, kv, batch, sc = device_objects(w, inp, DEV)
    sel = ops.SelectConfig(window_size=w.window_size)
    raw, ws = ops.score_paged(kv, batch, sc)
    keep_a, _ = ops.select(kv, batch, sc, sel, raw, ws)
    ops.compact(kv, batch, keep_a)
    torch.cuda.synchronize()
    chained = [c.clone() for c in caches]
    caches2, kv2, batch2, sc2 = device_objects(w, inp, DEV)
    keep_b, _ = ops.compress_step(kv2, batch2, sc2, sel)
    torch.cuda.synchronize()
    for b, t in enumerate(w.seq_lens):
        k = min(w.budget, t)
        rows = slice(b * w.num_kv_heads, (b + 1) * w.num_kv_heads)
        assert torch.equal(keep_a[rows, :k], keep_b[rows, :k])
    for a, b in zip(chained, caches2):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))


def test_end_to_end_c0_against_oracle():
    """One layer, one sequence of 4096 tokens: score, select at budget 2048, compact; kept K/V bit-exact."""
    w = synth.config(0)
    inp = build_inputs(w)
    caches, kv, batch, sc = device_objects(w, inp, DEV)
    sel = ops.SelectConfig(window_size=w.window_size)
    keep, _ = ops.compress_step(kv, batch, sc, sel)
    torch.cuda.synchronize()
    t, k, h = w.seq_lens[0], w.budget, w.num_kv_heads
    oraw = oracle_raw(w, inp, 0, t)
    okw = dict(window_size=w.window_size, chunk_tokens=osel.score_chunk_tokens(w.block_size, t))
    want, ofin = osel.group_keep_per_head(oraw, h, k, **okw)
    got = keep.cpu().long()
    fin64, bound = exact_gate(oraw, h, **okw)
    swapped = assert_keep_within_exact_bound(got, want, fin64, k, bound)
    record_swaps("c0_vs_oracle", swapped, h * k)
    assert swapped == 0
    # compaction is bit-exact given the device's own keep set
    ref = inp["caches"][0].clone()
    ocp.compact_per_head(ref, inp["tables"][0], w.block_size, got, t, full_permutation=False)
    blk, off = ocp.token_slots(inp["tables"][0], w.block_size, torch.arange(k))
    dev = caches[0].cpu()
    assert torch.equal(dev[:, blk, off].view(torch.int16), ref[:, blk, off].view(torch.int16))


RESIDENT_CASES = {
    "gqa4": dict(w=small()),
    "ragged": dict(w=small(seq_lens=(300, 17, 1000, 256, 513, 1), num_layers=3)),
    "hkv8": dict(w=small(num_q_heads=32, num_kv_heads=8, seq_lens=(700, 90), num_layers=4)),
    "hkv5_g3": dict(w=small(num_q_heads=15, num_kv_heads=5, seq_lens=(333, 130))),
    "hkv16": dict(w=small(num_q_heads=32, num_kv_heads=16, seq_lens=(450,))),
    "hkv32_g1": dict(w=small(num_q_heads=32, num_kv_heads=32, seq_lens=(200, 77))),
    "g1": dict(w=small(num_q_heads=2, num_kv_heads=2, seq_lens=(129,))),
    "g8": dict(w=small(num_q_heads=64, num_kv_heads=8, seq_lens=(700, 90), num_layers=3)),
    "g6_hkv3": dict(w=small(num_q_heads=18, num_kv_heads=3, seq_lens=(333, 130))),
    "g8_fp8_long": dict(w=small(kv_dtype="fp8", num_q_heads=16, num_kv_heads=2, seq_lens=(9000, 2500), budget=512)),
    "interleaved": dict(w=small(rope_style="interleaved")),
    "fp16": dict(w=small(kv_dtype="fp16")),
    "fp16_interleaved_ragged": dict(w=small(kv_dtype="fp16", rope_style="interleaved", seq_lens=(300, 17, 1000, 513),
                                            num_layers=3)),
    "fp16_g8": dict(w=small(kv_dtype="fp16", num_q_heads=16, num_kv_heads=2, seq_lens=(700, 90))),
    "fp16_tile192": dict(w=small(kv_dtype="fp16", seq_lens=(3072,) * 16, budget=256, num_layers=2)),
    "fp8": dict(w=small(kv_dtype="fp8", seq_lens=(300, 45))),
    "fp8_interleaved_hkv8": dict(w=small(kv_dtype="fp8", rope_style="interleaved", num_q_heads=32, num_kv_heads=8,
                                         seq_lens=(530, 64))),
    "block4": dict(w=small(block_size=4, seq_lens=(301,))),
    "block64": dict(w=small(block_size=64, seq_lens=(500, 31))),
    "kv_axis1": dict(w=small(seq_lens=(290, 64)), kv_axis=1),
    "one_layer": dict(w=small(num_layers=1)),
    "layer_max_group_mean": dict(w=small(num_layers=3), sel=dict(layer_reduce="max", group_reduce="mean")),
    "no_normalize": dict(w=small(), sel=dict(normalize=False)),
    "prefill_guard": dict(w=small(seq_lens=(400, 90)), sel=dict(protect_prefill=True), prefill_lens=[37, 5]),
    "tile320": dict(w=small(seq_lens=(2176,) * 30 + (1700, 33), budget=256, num_layers=2)),
    "tile256_fp8": dict(w=small(kv_dtype="fp8", seq_lens=(3000,) * 15 + (2990,), budget=256, num_layers=2)),
    "tw64": dict(w=small(seq_lens=(9000,) * 20, budget=512, num_layers=2)),
    "tw128": dict(w=small(seq_lens=(40000, 3000, 25001), budget=2048, num_layers=2)),
    "two_launches": dict(w=small(seq_lens=(70000, 100, 66000, 69000), budget=1024, num_layers=2)),
    "packed_ragged_launches": dict(w=small(seq_lens=(30000, 700, 61000, 9000, 45000, 1, 33000, 12000, 52000, 2100),
                                           budget=512, num_layers=2)),
}


# The same machinery with eight KV heads (workgroups of eight waves; the cases above mostly have
# two KV heads, which take workgroups of four waves, two per CU) on a device that pretends to
# hold 24 workgroups, so that small inputs need several, device-packed launches.
RESIDENT_CASES.update({
    "hkv8_ragged_small_chip": dict(w=small(num_q_heads=32, num_kv_heads=8, seq_lens=(3000, 70, 6100, 900, 4500, 1, 3300),
                                           budget=128, num_layers=2), workgroups=24),
    "hkv8_g8_small_chip": dict(w=small(num_q_heads=64, num_kv_heads=8, seq_lens=(2500, 300, 4000), budget=128,
                                       num_layers=2), workgroups=24),
    "hkv2_ragged_small_chip": dict(w=small(seq_lens=(3000, 70, 6100, 900, 4500, 1, 3300), budget=128, num_layers=2),
                                   workgroups=12),
    "hkv4_g7": dict(w=small(num_q_heads=28, num_kv_heads=4, seq_lens=(700, 90, 2049), num_layers=3)),
    "hkv4_g7_fp8": dict(w=small(kv_dtype="fp8", num_q_heads=28, num_kv_heads=4, seq_lens=(700, 1300))),
    "hkv3_fp16": dict(w=small(kv_dtype="fp16", num_q_heads=12, num_kv_heads=3, seq_lens=(640, 77))),
    # head dimension 64 (GPT-OSS: 64 query / 8 KV heads)
    "d64_g8_hkv8": dict(w=small(head_dim=64, num_q_heads=64, num_kv_heads=8, seq_lens=(700, 90, 1500), num_layers=3)),
    "d64_g4_hkv8_ragged_small_chip": dict(w=small(head_dim=64, num_q_heads=32, num_kv_heads=8,
                                                  seq_lens=(3000, 70, 6100, 900, 4500, 1), budget=128, num_layers=2),
                                          workgroups=24),
    "d64_hkv2": dict(w=small(head_dim=64, seq_lens=(300, 1000, 17))),
    "d64_interleaved_fp16_g7": dict(w=small(head_dim=64, kv_dtype="fp16", rope_style="interleaved", num_q_heads=28,
                                            num_kv_heads=4, seq_lens=(640, 2049))),
    # head dimension 256
    "d256_hkv8": dict(w=small(head_dim=256, num_q_heads=16, num_kv_heads=8, seq_lens=(700, 90, 1500), num_layers=3)),
    "d256_g8_fp16_interleaved": dict(w=small(head_dim=256, kv_dtype="fp16", rope_style="interleaved", num_q_heads=16,
                                             num_kv_heads=2, seq_lens=(640, 2049))),
    "d256_ragged_small_chip": dict(w=small(head_dim=256, num_q_heads=8, num_kv_heads=8,
                                           seq_lens=(3000, 70, 4100, 900, 1), budget=128, num_layers=2), workgroups=24),
    "d64_tile_refined": dict(w=small(head_dim=64, num_q_heads=32, num_kv_heads=8, seq_lens=(3072,) * 16, budget=256,
                                     num_layers=2)),
})


# Five to eight query heads, eight waves: the slack of a tile of 512 ends inside a rotation of the step buffers (seven steps), and a
# wave's sums pass through the ring slots behind its tile.  Whole tiles of 512, last tiles of one step, of the slack's seven and of
# one more.  Shorter tiles have more slack than a layer has steps: 128 on the short ring (below: 256), 320 with four waves.
RESIDENT_CASES.update({
    "g8_slack_whole_tiles_small_chip": dict(w=small(num_q_heads=64, num_kv_heads=8, budget=128, num_layers=3,
                                                    seq_lens=(12288, 10241, 5232, 4721, 113, 16)), workgroups=24,
                                            plan=dict(tile_tokens=512)),
    "g8_fp8_whole_tiles_small_chip": dict(w=small(num_q_heads=64, num_kv_heads=8, budget=128, num_layers=3, kv_dtype="fp8",
                                                  seq_lens=(12288, 10241, 5232, 4721, 113, 16)), workgroups=24,
                                          plan=dict(tile_tokens=512)),
    "g8_slack_short_ring": dict(w=small(num_q_heads=48, num_kv_heads=8, budget=128, num_layers=3,
                                        seq_lens=(256, 272, 369, 129, 1)), plan=dict(tile_tokens=128)),
    "g5_slack_hkv3": dict(w=small(num_q_heads=15, num_kv_heads=3, budget=128, num_layers=3,
                                  seq_lens=(6144, 5121, 640, 17)), workgroups=12, plan=dict(tile_tokens=320)),
})


# The same with at most four KV heads (workgroups of four waves, a device that holds 24 of them): sums that meet in LDS up to
# seven query heads, every wave's own with eight.  Tiles of 512, as "plan" says: the longest sequence leaves room for no other.
# Whole tiles, behind which the slack is four or five steps, and last tiles of 1, 4, 5 and 6 steps.
FOUR_WAVES = dict(budget=128, num_layers=3, seq_lens=(12288, 10241, 5200, 4689, 4672, 1088, 16))
for tag, heads, more in [("g5_hkv3", (15, 3), {}), ("g6_hkv4", (24, 4), dict(rope_style="interleaved")), ("g7_hkv4", (28, 4), {}),
                         ("g8_hkv2", (16, 2), {}), ("g7_hkv2_fp16", (14, 2), dict(kv_dtype="fp16")),
                         ("g7_hkv4_fp8", (28, 4), dict(kv_dtype="fp8")), ("g8_hkv1_fp8", (8, 1), dict(kv_dtype="fp8")),
                         ("d64_g7_hkv4", (28, 4), dict(head_dim=64)), ("d64_g8_hkv2", (16, 2), dict(head_dim=64)),
                         ("d256_g5_hkv2", (10, 2), dict(head_dim=256))]:
    RESIDENT_CASES["four_waves_" + tag] = dict(w=small(num_q_heads=heads[0], num_kv_heads=heads[1], **FOUR_WAVES, **more),
                                               workgroups=12, plan=dict(tile_tokens=512))

# Tiles of 256 on the short ring of five to eight query heads: whole ones, last ones of 1, 4 and 15 steps.
for tag, heads, more in [("g6", (48, 8), {}), ("g8_fp16", (64, 8), dict(kv_dtype="fp16")), ("g8_fp8", (64, 8), dict(kv_dtype="fp8"))]:
    RESIDENT_CASES["short_ring_" + tag] = dict(w=small(num_q_heads=heads[0], num_kv_heads=heads[1], budget=128, num_layers=3,
                                                       seq_lens=(1536, 1281, 1344, 1520), **more),
                                               workgroups=24, plan=dict(tile_tokens=256, launches=1))


@pytest.mark.parametrize("case", ["one_request_36_layers", "one_request_split_by_layer", "one_request_uneven_layer_groups",
                                  "three_requests_split", "sixteen_requests"])
def test_steady_state_step_matches_oracle(case, monkeypatch):
    """The step a long generation repeats every 128 tokens: budget + 128 = 2176 cached tokens, budget
    2048, Qwen3-8B head shape, against the CPU oracle: kept sets, and K/V compacted bit for bit.
    One request (what the reference's runner hands over, runtime/runner_compression_actions.py:24)
    does not fill the chip with whole-model workgroups; the resident kernel then cuts the layers
    into groups.  Sixteen requests run as whole-model workgroups."""
    layers, seqs, env = {
        "one_request_36_layers": (36, 1, {}),                                   # the library's own choice
        "one_request_split_by_layer": (4, 1, {"TRIATTN_RESIDENT_KERNEL": "mfma", "TRIATTN_RESIDENT_LAYER_SPLIT": "1"}),
        "one_request_uneven_layer_groups": (5, 1, {"TRIATTN_RESIDENT_KERNEL": "mfma", "TRIATTN_RESIDENT_LAYER_SPLIT": "1",
                                                   "TRIATTN_RESIDENT_WORKGROUPS": "12"}),    # groups of 2, 2, 1 layers
        "three_requests_split": (6, 3, {"TRIATTN_RESIDENT_KERNEL": "mfma", "TRIATTN_RESIDENT_LAYER_SPLIT": "1",
                                        "TRIATTN_RESIDENT_WORKGROUPS": "40"}),
        "sixteen_requests": (4, 16, {}),
    }[case]
    tune(**env)
    w = synth.Workload("steady", layers, 32, 8, 128, (2176,) * seqs, 2048, index=70 + layers)
    inp = build_inputs(w)
    caches, kv, batch, sc = device_objects(w, inp, DEV)
    sel = ops.SelectConfig(window_size=w.window_size)
    assert ops.select_path(kv, batch, sc, sel) == "resident_mfma"
    _, fin, ws = ops.select_paged(kv, batch, sc, sel, want_scores=True)
    keep, ws = ops.compress_step(kv, batch, sc, sel, ws)
    assert ws.status() == 0
    keep, fin = keep.cpu().long(), fin.cpu()
    h, k, t = w.num_kv_heads, w.budget, 2176
    swapped = 0
    for b in range(seqs):
        oraw = oracle_raw(w, inp, b, t)
        okw = dict(window_size=w.window_size, chunk_tokens=osel.score_chunk_tokens(w.block_size, t))
        want, ofin = osel.group_keep_per_head(oraw, h, k, **okw)
        finite = torch.isfinite(ofin)
        scale = float(ofin[finite].abs().max())
        dfin = fin[b * h:(b + 1) * h, :t]
        assert torch.equal(torch.isfinite(dfin), finite)
        assert float((dfin[finite] - ofin[finite]).abs().max()) <= selection_score_tol(oraw) * scale
        got = keep[b * h:(b + 1) * h, :k]
        fin64, bound = exact_gate(oraw, h, **okw)
        swapped += assert_keep_within_exact_bound(got, want, fin64, k, bound)
        blk, off = ocp.token_slots(inp["tables"][b], w.block_size, torch.arange(k))
        for l in range(0, layers, max(1, layers // 4)):
            ref = inp["caches"][l].clone()
            ocp.compact_per_head(ref, inp["tables"][b], w.block_size, got, t, full_permutation=False)
            assert torch.equal(caches[l].cpu()[:, blk, off].view(torch.int16), ref[:, blk, off].view(torch.int16)), (b, l)
    record_swaps(f"steady_state_vs_oracle:{case}", swapped, seqs * h * k)


# Named cases in which the two paths keep different indices at near-ties (scores within
# KEEP_TIE_TOL of the threshold), and how many of the case's kept indices: 16 sequences x heads x
# 256 kept indices each, two of which sit that close to their threshold.  Everywhere else: none.
# (four_waves_d256_g5_hkv2 and short_ring_g6: one pair of 1568 and of 4096 kept indices, within the exact bound asserted below, and
# the same pair whichever way the sums of a layer are published and whatever the slack: the bits do not depend on either.)
NEAR_TIES = {("fp16_tile192", "mfma"): 2, ("d64_tile_refined", "mfma"): 2, ("four_waves_d256_g5_hkv2", "mfma"): 2,
              ("short_ring_g6", "mfma"): 2}


@pytest.mark.parametrize("kernel", ["mfma", "valu"])
@pytest.mark.parametrize("name", list(RESIDENT_CASES))
def test_resident_selection_matches_two_pass(name, kernel, monkeypatch):
    """The single resident kernel (raw scores kept in LDS) against score_paged + select:
    same selection scores up to the rounding of differently grouped fp32 sums in the
    statistics (the reference's streaming variance sumsq - n*mean^2 amplifies that
    rounding by mean^2/var), same kept sets away from ties."""
    case = dict(RESIDENT_CASES[name])
    w = case["w"]
    if kernel == "mfma" and w.block_size < 16:
        pytest.skip("the matrix-core kernel needs blocks of at least 16 tokens (a step lies inside one block)")
    if kernel == "valu" and w.num_q_heads // w.num_kv_heads > 4:
        pytest.skip("the vector-unit kernel holds four query heads per KV head")
    if kernel == "valu" and w.head_dim != 128:      # (64 and 256 exist on the matrix cores only)
        pytest.skip("the vector-unit kernel is built for a head dimension of 128")
    tune(resident_kernel=kernel)      # take that kernel however small the launch
    if "workgroups" in case:
        tune(resident_workgroups=case["workgroups"])
    if "layer_split" in case:
        tune(layer_split=case["layer_split"])
    inp = build_inputs(w, case.get("kv_axis", 0))
    print(f"case={name} kernel={kernel} workload={w}", flush=True)
    caches, kv, batch, sc = device_objects(w, inp, DEV, prefill_lens=case.get("prefill_lens"))
    selkw = dict(window_size=w.window_size)
    selkw.update(case.get("sel", {}))
    sel = ops.SelectConfig(**selkw)
    assert ops.select_path(kv, batch, sc, sel) == "resident_" + kernel
    if "plan" in case:                # what the case is there for
        plan = ops.describe_plan(kv, batch, sc, sel)
        assert {key: plan[key] for key in case["plan"]} == case["plan"], plan
    keep_r, fin_r, ws = ops.select_paged(kv, batch, sc, sel, want_scores=True)
    raw, ws2 = ops.score_paged(kv, batch, sc)
    keep_t, fin_t = ops.select(kv, batch, sc, sel, raw, ws2, want_scores=True)
    torch.cuda.synchronize()
    assert ws.status() == 0
    h = w.num_kv_heads
    swapped = compared = 0
    for b, t in enumerate(w.seq_lens):
        k = min(w.budget, t)
        fr, ft = fin_r[b * h:(b + 1) * h, :t].cpu(), fin_t[b * h:(b + 1) * h, :t].cpu()
        assert torch.equal(torch.isinf(fr), torch.isinf(ft))
        finite = torch.isfinite(ft)
        scale = float(ft[finite].abs().max()) if bool(finite.any()) else 1.0
        tol = selection_score_tol(raw[b, :, :t].transpose(-1, -2).cpu()) if sel.normalize else SELECT_SCORE_TOL
        assert float((fr[finite] - ft[finite]).abs().max() if bool(finite.any()) else 0.0) <= tol * scale, (name, b)
        rows_r, rows_t = keep_r[b * h:(b + 1) * h, :k].cpu().long(), keep_t[b * h:(b + 1) * h, :k].cpu().long()
        if sel.group_reduce == "max" and k < t and bool(finite.any()):
            # Both against the exact evaluation of the reference's formula on the two-pass raw scores:
            # an index may differ only where an fp32 evaluation of that formula is itself undecided.
            prefill = case.get("prefill_lens")
            _, fin64, bound = device_exact_gate(raw, b, t, h, k, w.block_size, normalize=bool(sel.normalize),
                                                window_size=sel.window_size, protect_prefill=sel.protect_prefill,
                                                prefill_len=prefill[b] if prefill else 0, layer_agg=sel.layer_reduce)
            swapped += assert_keep_within_exact_bound(rows_r, rows_t, fin64, k, max(bound, 2.0 ** -22 * scale))
        else:
            swapped += assert_keep_matches(rows_r, rows_t, ft, k, tie_tol=KEEP_TIE_TOL * scale)
        compared += h * k
    record_swaps(f"resident_{kernel}_vs_two_pass:{name}", swapped, compared)
    if not name.startswith("random"):
        assert swapped <= NEAR_TIES.get((name, kernel), 0), (name, kernel, swapped)


def _random_resident_case(seed: int):
    """A seeded random shape the matrix-core kernel has an instance for."""
    import random
    r = random.Random(seed)
    kv_dtype = r.choice(["bf16", "bf16", "fp16", "fp8"])
    head_dim = 128 if kv_dtype == "fp8" else r.choice([128, 128, 64, 256])
    hkv = r.choice([1, 2, 3, 4, 5, 8, 8, 12])
    g = r.choice([1, 2, 3, 4, 4, 6, 7, 8])
    nseq = r.choice([1, 2, 3, 5, 9])
    seq_lens = tuple(r.choice([1, 15, 16, 17, 63, 64, 65, 127, 129, 300, 511, 513, 1023, 1025, 2049, 3000])
                     for _ in range(nseq))
    layers = r.choice([1, 2, 3])
    r2 = random.Random(10_000 + seed)           # (drawn apart, so that the other fields of a seed stay what they were)
    split = r2.random() < 0.5                   # let the planner cut the layers into groups of workgroups
    if split:
        layers = r2.choice([2, 3, 4, 5, 6, 7])
    w = small(kv_dtype=kv_dtype, head_dim=head_dim, num_q_heads=hkv * g, num_kv_heads=hkv, seq_lens=seq_lens,
              num_layers=layers, budget=r.choice([1, 16, 96, 200]), block_size=r.choice([16, 16, 32, 128]),
              window_size=r.choice([0, 1, 12, 200]), rope_style=r.choice(["half", "interleaved"]), index=100 + seed)
    case = dict(w=w, sel=dict(normalize=r.random() < 0.8, group_reduce=r.choice(["max", "max", "mean"]),
                              layer_reduce=r.choice(["mean", "mean", "max"])))
    if r.random() < 0.3:
        case["sel"]["protect_prefill"] = True
        case["prefill_lens"] = [r.randrange(0, t + 1) for t in seq_lens]
    if r.random() < 0.4:
        case["workgroups"] = r.choice([16, 24, 40])      # enough for the longest sequence at its smallest tile
    if split:
        case["layer_split"] = 1
    return case


@pytest.mark.parametrize("seed", range(int(os.environ.get("TRIATTN_TEST_RANDOM_SHAPES", "32"))))
def test_matrix_core_kernel_on_random_shapes(seed, monkeypatch):
    """Seeded random head layouts, key types, head dimensions, ragged lengths, block sizes, guards
    and device sizes: resident matrix-core selection against the two-pass kernels."""
    case = _random_resident_case(seed)
    RESIDENT_CASES[f"random{seed}"] = case
    try:
        test_resident_selection_matches_two_pass(f"random{seed}", "mfma", monkeypatch)
    finally:
        del RESIDENT_CASES[f"random{seed}"]


@pytest.mark.parametrize("kv_dtype,head_dim", [("bf16", 128), ("fp16", 128), ("fp8", 128), ("bf16", 64), ("fp16", 64),
                                               ("bf16", 256), ("fp16", 256)])
def test_matrix_core_scores_carry_every_piece(kv_dtype, head_dim, monkeypatch):
    """Without normalisation and with a layer maximum the raw scores show through: the
    matrix-core kernel (coefficients in three pieces, magnitudes in two) agrees with the
    two-pass kernels' fp32 arithmetic to 5e-6 of the largest score (measured: 2e-7 .. 1.5e-6);
    a dropped second piece of the magnitudes would show as 1e-4 .. 2e-3."""
    w = small(kv_dtype=kv_dtype, head_dim=head_dim, seq_lens=(3000, 1000), index=77)
    _assert_scores_carry_every_piece(w)


@pytest.mark.parametrize("kv_dtype,head_dim,g", [("bf16", 128, 5), ("bf16", 64, 8), ("bf16", 256, 7), ("fp16", 128, 8),
                                                 ("fp16", 64, 6), ("fp8", 128, 8)])
def test_every_piece_of_five_to_eight_query_heads(kv_dtype, head_dim, g, monkeypatch):
    """The operand layout of five to eight query heads per KV head (two pieces side by side, the third in an
    operand of its own, of the magnitude coefficients too): same bound as with four.  Tiles that end
    inside a step, one token into it and at its end."""
    w = small(kv_dtype=kv_dtype, head_dim=head_dim, num_q_heads=3 * g, num_kv_heads=3, seq_lens=(1201, 1000, 33), index=78)
    _assert_scores_carry_every_piece(w)


def _assert_scores_carry_every_piece(w):
    kv_dtype, head_dim = w.kv_dtype, w.head_dim
    inp = build_inputs(w)
    caches, kv, batch, sc = device_objects(w, inp, DEV)
    sel = ops.SelectConfig(window_size=w.window_size, normalize=False, layer_reduce="max")
    tune(resident_kernel="mfma")
    assert ops.select_path(kv, batch, sc, sel) == "resident_mfma"
    _, fin_r, ws = ops.select_paged(kv, batch, sc, sel, want_scores=True)
    tune(resident_kernel="off")
    _, fin_t, _ = ops.select_paged(kv, batch, sc, sel, want_scores=True)
    torch.cuda.synchronize()
    assert ws.status() == 0
    h = w.num_kv_heads
    for b, t in enumerate(w.seq_lens):
        a, c = fin_r[b * h:(b + 1) * h, :t], fin_t[b * h:(b + 1) * h, :t]
        m = torch.isfinite(c)
        assert float((a[m] - c[m]).abs().max()) <= 5e-6 * float(c[m].abs().max()), (kv_dtype, head_dim, b)


@pytest.mark.parametrize("kernel", ["mfma", "valu"])
def test_resident_selection_on_dense_keys(kernel, monkeypatch):
    """[B, H, T, D] keys without a block table (the selector's keys_dense call shape) through
    the resident kernels: the 'block' of a sequence is the sequence itself."""
    g = torch.Generator().manual_seed(11)
    b, hkv, hq, t, d = 3, 4, 8, 700, 128
    keys = (torch.randn(b, hkv, t, d, generator=g) + torch.randn(1, hkv, 1, d, generator=g)).to(torch.bfloat16).to(DEV)
    qc = torch.randn(2, hq, d // 2, 2, generator=g)
    qa = qc.pow(2).sum(-1).sqrt() + torch.rand(2, hq, d // 2, generator=g)
    sc = ops.ScoreConfig(ops.fold_stats(qc.to(DEV), qa.to(DEV), torch.ones_like(qa).to(DEV)),
                         synth.rope_inv_freq(small()).to(DEV), synth.geometric_offsets().to(DEV))
    # two "layers" that share the key tensor (a PagedKV of dense keys holds one view per layer)
    view = keys.permute(0, 2, 1, 3)
    kv = ops.PagedKV([view, view], None)
    lens = [t, 333, 512]
    batch = ops.StepBatch(DEV, lens, round_start=[900, 400, 512], budgets=128)
    sel = ops.SelectConfig(window_size=16)
    print(f"dense keys kernel={kernel}", flush=True)
    tune(resident_kernel=kernel)
    assert ops.select_path(kv, batch, sc, sel) == "resident_" + kernel
    keep_r, fin_r, ws = ops.select_paged(kv, batch, sc, sel, want_scores=True)
    torch.cuda.synchronize()
    assert ws.status() == 0
    tune(resident_kernel="off")
    assert ops.select_path(kv, batch, sc, sel) == "two_pass"
    keep_t, fin_t, _ = ops.select_paged(kv, batch, sc, sel, want_scores=True)
    torch.cuda.synchronize()
    for i, n in enumerate(lens):
        fr, ft = fin_r[i * hkv:(i + 1) * hkv, :n].cpu(), fin_t[i * hkv:(i + 1) * hkv, :n].cpu()
        assert torch.equal(torch.isinf(fr), torch.isinf(ft))
        finite = torch.isfinite(ft)
        scale = float(ft[finite].abs().max())
        assert float((fr[finite] - ft[finite]).abs().max()) <= 5e-4 * scale
        assert_keep_matches(keep_r[i * hkv:(i + 1) * hkv, :128].cpu().long(), keep_t[i * hkv:(i + 1) * hkv, :128].cpu().long(),
                            ft, 128, tie_tol=2e-3 * scale)


def test_resident_path_is_taken_unless_multi_layer_workgroups_would_underfill_the_chip():
    """Workgroups that run one layer make a short launch however few they are; workgroups that run
    several layers must fill most of the chip, or the two-pass kernels take the batch.  Of the short ones the smallest
    are two launches of their own under the automatic choice; the plan says so beside the resident one's cut."""
    sel = ops.SelectConfig(window_size=12)
    cases = ((1, None, (300,), "resident_mfma"),             # 3 tiles of 128, one layer
             (1, None, (16384,), "resident_mfma"),           # 64 tiles, a quarter of the chip, one layer
             (1, None, (2176,) * 4, "resident_mfma"),
             (4, None, (300,), "resident_mfma"),             # cut into 4 layer groups x 3 tiles
             (4, 0, (300,), "two_pass"),                     # layer groups switched off: 3 workgroups x 4 layers
             (4, 0, (2176,) * 4, "two_pass"),                # 4 x 17 tiles of 128 x 4 layers
             (4, 0, (8192,) * 4, "resident_mfma"),           # 4 x 64 tiles of 128: the chip is full
             (4, None, (128,) * 130, "two_pass"),            # 130 workgroups, two layer groups would not fit
             (1, None, (3072,) * 16, "resident_mfma"), (1, None, (2176,) * 16, "resident_mfma"))
    for layers, split, seq_lens, want in cases:
        tune(layer_split=-1 if split is None else split)
        w = small(seq_lens=seq_lens, num_layers=layers, num_q_heads=32, num_kv_heads=8)
        tables = synth.make_block_tables(w)
        cache = torch.zeros(2, w.pool_blocks, w.block_size, w.num_kv_heads, w.head_dim, dtype=torch.bfloat16, device=DEV)
        kv = ops.PagedKV.from_kv_caches([cache] * layers)
        batch = ops.StepBatch(DEV, w.seq_lens, round_start=w.seq_lens, budgets=w.budget, block_tables=tables)
        qc, qa = synth.make_stats(w, DEV)
        sc = ops.ScoreConfig(ops.fold_stats(qc, qa, torch.ones_like(qa)), synth.rope_inv_freq(w, DEV),
                             synth.geometric_offsets(device=DEV))
        assert ops.select_path(kv, batch, sc, sel) == want, (layers, split, seq_lens)
        info = ops.describe_plan(kv, batch, sc, sel)
        assert info["path"] == want
        if want != "two_pass":
            assert info["small_launches"] == (layers * len(seq_lens) * 8 * -(-max(seq_lens) // 128) <= 1024
                                              and max(seq_lens) <= 8192)
            # the dry run for a device of this one's size gives this device's plan, and a launch fits the device
            assert ops.describe_plan(kv, batch, sc, sel, assume_resident_workgroups=info["resident_workgroups"]) == info
            assert info["launches"] == 1 and info["layer_groups"] * info["layers_per_group"] >= layers
            assert len(seq_lens) * info["layer_groups"] * info["tiles_per_seq"] <= info["resident_workgroups"]


def _resident_batch(seed_index):
    w = small(seq_lens=(3072,) * 16, num_layers=2, budget=256, index=seed_index)
    inp = build_inputs(w)
    caches, kv, batch, sc = device_objects(w, inp, DEV)
    return w, inp, caches, kv, batch, sc


def test_resident_launches_on_two_streams_do_not_starve_each_other():
    """Each launch wants most of the CUs; issued from two streams at once they are chained on
    the device, so both finish with a clean status and the same result as alone."""
    sel = ops.SelectConfig(window_size=12)
    jobs = [_resident_batch(11), _resident_batch(12)]
    alone = []
    for w, inp, caches, kv, batch, sc in jobs:
        assert ops.select_path(kv, batch, sc, sel) == "resident_mfma"
        keep, fin, ws = ops.select_paged(kv, batch, sc, sel, want_scores=True)
        assert ws.status() == 0
        alone.append((keep.clone(), fin.clone()))
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    outs = []
    for rep in range(3):
        for (w, inp, caches, kv, batch, sc), st in zip(jobs, streams):
            with torch.cuda.stream(st):
                outs.append(ops.select_paged(kv, batch, sc, sel, want_scores=True))
    torch.cuda.synchronize()
    for i, (keep, fin, ws) in enumerate(outs):
        assert ws.status() == 0
        assert torch.equal(keep, alone[i % 2][0]) and torch.equal(fin, alone[i % 2][1])


def test_resident_launch_next_to_another_streams_kernels():
    """A serving process keeps the GPU busy with its own kernels on other streams.  The resident
    launch assumes that all its workgroups reach a CU; another stream's kernels only delay that
    (they end), so steps issued while a second stream runs a queue of large matrix products finish
    with a clean status and the same keep rows and caches as on an idle GPU."""
    sel = ops.SelectConfig(window_size=12)
    w, inp, caches, kv, batch, sc = _resident_batch(13)
    assert ops.select_path(kv, batch, sc, sel) == "resident_mfma"
    pristine = [c.clone() for c in caches]
    keep0, ws = ops.compress_step(kv, batch, sc, sel)
    assert ws.status() == 0
    want = [c.clone() for c in caches]
    side = torch.cuda.Stream()
    a = torch.randn(6144, 6144, device=DEV, dtype=torch.bfloat16)
    out = torch.empty_like(a)
    torch.cuda.synchronize()
    print("steps next to a queue of matrix products", flush=True)
    for rep in range(4):
        for c, p in zip(caches, pristine):
            c.copy_(p)
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            for _ in range(60):
                torch.matmul(a, a, out=out)
        keep = torch.empty_like(keep0)
        ops.compress_step(kv, batch, sc, sel, ws, keep)      # queued while the products run
        torch.cuda.synchronize()
        assert ws.status() == 0, f"repetition {rep}"
        assert torch.equal(keep, keep0)
        for c, x in zip(caches, want):
            assert torch.equal(c.view(torch.int16), x.view(torch.int16))


def test_replayed_resident_graph_is_chained_with_eager_resident_launches():
    """A captured step holds no wait on the process's previous resident launch and no record of its
    own (streams under capture are left alone).  Whoever replays such a graph brackets the replay with
    ops.resident_gate(); replays on one stream then interleave with eager resident launches on another
    without either starving the other: clean status words, the results of running alone."""
    sel = ops.SelectConfig(window_size=12)
    w1, inp1, caches1, kv1, batch1, sc1 = _resident_batch(21)
    w2, inp2, caches2, kv2, batch2, sc2 = _resident_batch(22)
    for kv, batch, sc in ((kv1, batch1, sc1), (kv2, batch2, sc2)):
        assert ops.select_path(kv, batch, sc, sel) == "resident_mfma"
    keep_a, fin_a, ws_a = ops.select_paged(kv1, batch1, sc1, sel, want_scores=True)
    keep_b, fin_b, ws_b = ops.select_paged(kv2, batch2, sc2, sel, want_scores=True)
    assert ws_a.status() == 0 and ws_b.status() == 0
    want_a, want_b = (keep_a.clone(), fin_a.clone()), (keep_b.clone(), fin_b.clone())
    s_graph, s_eager = torch.cuda.Stream(), torch.cuda.Stream()
    s_graph.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s_graph):
        ops.select_paged(kv1, batch1, sc1, sel, ws_a, keep=keep_a, scores_out=fin_a)     # warm-up on the capture stream
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s_graph):
        ops.select_paged(kv1, batch1, sc1, sel, ws_a, keep=keep_a, scores_out=fin_a)
    print("replays next to eager resident launches", flush=True)
    for rep in range(4):
        keep_a.zero_(); fin_a.zero_(); keep_b.zero_(); fin_b.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(s_eager):
            ops.select_paged(kv2, batch2, sc2, sel, ws_b, keep=keep_b, scores_out=fin_b)
        with torch.cuda.stream(s_graph):
            with ops.resident_gate():
                graph.replay()
        with torch.cuda.stream(s_eager):
            ops.select_paged(kv2, batch2, sc2, sel, ws_b, keep=keep_b, scores_out=fin_b)
        with torch.cuda.stream(s_graph):
            with ops.resident_gate():
                graph.replay()
        torch.cuda.synchronize()
        assert ws_a.status() == 0 and ws_b.status() == 0, rep
        assert torch.equal(keep_a, want_a[0]) and torch.equal(fin_a, want_a[1]), rep
        assert torch.equal(keep_b, want_b[0]) and torch.equal(fin_b, want_b[1]), rep


@pytest.mark.parametrize("case", ["fewer_launches_planned_than_needed", "device_length_beyond_max_seq_len"])
def test_host_lengths_that_disagree_with_the_device_raise_the_status_word(case, monkeypatch):
    """A caller of the C ABI whose host copy of the lengths is stale: the planner sizes launches
    and rows from the host values, the kernels read the device values.  Sequences that would not
    be scored (or lie beyond the planned rows) raise the status word (3), every workgroup still
    runs to its end inside the planned bounds, and the step's compaction leaves the cache alone."""
    tune(resident_kernel="mfma")
    if case == "fewer_launches_planned_than_needed":
        tune(resident_workgroups=16)
        w = small(seq_lens=(3000,) * 8, num_q_heads=32, num_kv_heads=8, budget=128, index=51)
    else:
        w = small(seq_lens=(1000, 700), num_q_heads=32, num_kv_heads=8, budget=128, index=52)
    inp = build_inputs(w)
    caches, kv, batch, sc = device_objects(w, inp, DEV)
    sel = ops.SelectConfig(window_size=w.window_size)
    keep, ws = ops.compress_step(kv, batch, sc, sel)            # lengths agree: a clean step
    assert ws.status() == 0
    caches, kv, batch, sc = device_objects(w, inp, DEV)
    pristine = [c.clone() for c in caches]
    if case == "fewer_launches_planned_than_needed":
        for i in range(1, w.num_seqs):
            batch._lens_host[i] = 100          # the host believes seven sequences are short: one launch planned
    else:
        batch.seq_lens[1] = 1500               # the device holds more than max_seq_len = 1000
    assert ops.select_path(kv, batch, sc, sel) == "resident_mfma"
    keep, ws = ops.compress_step(kv, batch, sc, sel)
    assert ws.status() == 3
    for c, p in zip(caches, pristine):
        assert torch.equal(c.view(torch.int16), p.view(torch.int16))


@pytest.mark.parametrize("kv_dtype", ["bf16", "fp8"])
def test_compress_step_replays_from_a_hip_graph(kv_dtype):
    """The launch sequence of a step (no allocation, no synchronisation, no memset nodes)
    captured once and replayed: every replay must equal the eager result.  With an fp8 cache
    the eager step moves the scales on the library's side stream, the captured one on the
    capture stream; the scale arrays are part of the comparison."""
    w = small(seq_lens=(3072,) * 16, num_layers=2, budget=256, index=13, kv_dtype=kv_dtype)
    inp = build_inputs(w)
    caches, kv, batch, sc = device_objects(w, inp, DEV)
    if kv_dtype == "fp8":
        caches = list(caches) + list(kv._keep[2]) + list(kv._keep[3])      # codes, K scales, V scales
    pristine = [c.clone() for c in caches]
    sel = ops.SelectConfig(window_size=12)
    ws = ops.Workspace(kv, batch, sc)
    keep = torch.empty(w.num_seqs * w.num_kv_heads, batch.max_budget, dtype=torch.int32, device=DEV)
    ops.compress_step(kv, batch, sc, sel, ws, keep)
    torch.cuda.synchronize()
    want_keep, want_caches = keep.clone(), [c.clone() for c in caches]

    def restore():
        for c, p in zip(caches, pristine):
            c.copy_(p)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        restore()
        ops.compress_step(kv, batch, sc, sel, ws, keep)      # warm-up on the capture stream
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    restore()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        ops.compress_step(kv, batch, sc, sel, ws, keep)
    for rep in range(3):
        restore()
        keep.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert ws.status() == 0
        assert torch.equal(keep, want_keep), rep
        for c, wc in zip(caches, want_caches):
            assert torch.equal(c.view(torch.uint8), wc.view(torch.uint8)), rep


@pytest.mark.parametrize("kernel", ["mfma", "valu"])
def test_expired_wait_raises_the_status_word_and_the_step_leaves_the_cache_alone(kernel, monkeypatch):
    """The resident kernels' failure path, forced from the host: with a negative wait limit every
    wait on another workgroup gives up at once, all workgroups still run to their end, the status
    word reads non-zero and the compaction of compress_step moves nothing.  The same call
    without the limit then gives the result of the chained calls."""
    w, inp, caches, kv, batch, sc = _resident_batch(21)
    sel = ops.SelectConfig(window_size=w.window_size)
    tune(resident_kernel=kernel)
    assert ops.select_path(kv, batch, sc, sel) == "resident_" + kernel
    before = [c.clone() for c in caches]
    tune(resident_wait_us=-1)
    print(f"forced expiry, kernel={kernel}", flush=True)
    _, ws = ops.compress_step(kv, batch, sc, sel)
    assert ws.status() != 0
    for c, c0 in zip(caches, before):
        assert torch.equal(c.view(torch.int16), c0.view(torch.int16))
    tune(resident_wait_us=None)
    keep, ws = ops.compress_step(kv, batch, sc, sel, ws=ws)
    assert ws.status() == 0
    caches2, kv2, batch2, sc2 = device_objects(w, inp, DEV)
    keep2, _, ws2 = ops.select_paged(kv2, batch2, sc2, sel)
    ops.compact(kv2, batch2, keep2)
    torch.cuda.synchronize()
    assert torch.equal(keep, keep2)
    for c, c2 in zip(caches, caches2):
        assert torch.equal(c.view(torch.int16), c2.view(torch.int16))


def test_fp16_coefficients_beyond_half_range_raise_the_status_word(monkeypatch):
    """The matrix-core kernel for fp16 keys holds its coefficients as fp16 pieces; statistics
    so large that a coefficient exceeds 65504 cannot be held, and the launch says so through
    the status word instead of returning scores made of infinities."""
    w = small(kv_dtype="fp16", seq_lens=(300, 200))
    inp = build_inputs(w)
    inp["qc"] = inp["qc"] * 1e6
    inp["qa"] = inp["qa"] * 1e6
    caches, kv, batch, sc = device_objects(w, inp, DEV)
    sel = ops.SelectConfig(window_size=w.window_size)
    tune(resident_kernel="mfma")
    assert ops.select_path(kv, batch, sc, sel) == "resident_mfma"
    print("fp16 coefficient overflow", flush=True)
    _, _, ws = ops.select_paged(kv, batch, sc, sel)
    assert ws.status() != 0
    tune(resident_kernel="valu")
    _, _, ws = ops.select_paged(kv, batch, sc, sel)
    assert ws.status() == 0


@pytest.mark.parametrize("what", ["key", "coefficient", "tiny_keys"])
def test_magnitudes_beyond_half_range_raise_the_status_word(monkeypatch, what):
    """Whatever the key type, the matrix-core kernel carries the magnitudes |k_f| and their
    coefficients as fp16 pieces.  A bf16 key whose magnitude exceeds 65504, statistics that make a
    magnitude coefficient that large, or keys so small throughout that their magnitudes are fp16
    subnormals (scaled by 2^-14) cannot be held: the launch raises the status word (2), the step
    moves nothing, and the same step on the other kernels gives the oracle's keep set."""
    w = small(seq_lens=(300, 200))
    inp = build_inputs(w)
    if what == "key":
        inp["caches"][1][0, int(inp["tables"][1][3]), 5, 1, 40] = 1.0e5     # K plane, one element of one row
    elif what == "tiny_keys":
        inp["caches"] = [(c.float() * 2.0 ** -14).to(c.dtype) for c in inp["caches"]]
    else:
        inp["qa"] = inp["qa"] * 1e6
    caches, kv, batch, sc = device_objects(w, inp, DEV)
    sel = ops.SelectConfig(window_size=w.window_size)
    tune(resident_kernel="mfma")
    assert ops.select_path(kv, batch, sc, sel) == "resident_mfma"
    print(f"magnitude overflow: {what}", flush=True)
    before = [c.clone() for c in caches]
    _, ws = ops.compress_step(kv, batch, sc, sel)
    assert ws.status() == 2
    for c, c0 in zip(caches, before):
        assert torch.equal(c.view(torch.int16), c0.view(torch.int16))
    for kernel in ("valu", "off"):
        tune(resident_kernel=kernel)
        keep, fin, ws = ops.select_paged(kv, batch, sc, sel, want_scores=True)
        assert ws.status() == 0 and bool(torch.isfinite(fin[0, :50]).all())
    keep = keep.cpu().long()
    h = w.num_kv_heads
    for b, t in enumerate(w.seq_lens):
        k = min(w.budget, t)
        oraw = oracle_raw(w, inp, b, t)
        want, ofin = osel.group_keep_per_head(oraw, h, w.budget, window_size=w.window_size,
                                              chunk_tokens=osel.score_chunk_tokens(w.block_size, t))
        scale = float(ofin[torch.isfinite(ofin)].abs().max())
        assert_keep_matches(keep[b * h:(b + 1) * h, :k], want, ofin, k, tie_tol=KEEP_TIE_TOL * scale)


def test_resident_path_falls_back_when_shape_has_no_kernel(monkeypatch):
    tune(resident_kernel="mfma")        # even when asked for explicitly
    for kw, selkw in ((dict(num_q_heads=32, num_kv_heads=2), {}), (dict(head_dim=256, kv_dtype="fp8"), {}), (dict(head_dim=64, kv_dtype="fp8"), {}),
                      (dict(block_size=24), {}), ({}, dict(shared=True)), ({}, dict(layer_reduce=None))):
        w = small(**kw)
        inp = build_inputs(w)
        caches, kv, batch, sc = device_objects(w, inp, DEV)
        sel = ops.SelectConfig(window_size=w.window_size, **selkw)
        assert ops.select_path(kv, batch, sc, sel) == "two_pass", (kw, selkw)
        keep_a, fin_a, ws = ops.select_paged(kv, batch, sc, sel, want_scores=True)
        raw, ws2 = ops.score_paged(kv, batch, sc)
        keep_b, fin_b = ops.select(kv, batch, sc, sel, raw, ws2, want_scores=True)
        torch.cuda.synchronize()
        assert torch.equal(keep_a, keep_b) and torch.equal(fin_a[:, :300], fin_b[:, :300])


@pytest.mark.parametrize("kw", [
    dict(num_q_heads=32, num_kv_heads=8),
    dict(num_q_heads=24, num_kv_heads=8, block_size=1),
    dict(num_q_heads=10, num_kv_heads=5, head_dim=128, kv_dtype="fp8"),
    dict(num_q_heads=24, num_kv_heads=3, head_dim=256),
], ids=["gqa4", "token_blocks", "five_heads_fp8", "d256_gqa8"])
@pytest.mark.parametrize("lens", [(1,), (127, 2), (128, 129), (513, 31, 4), (511, 1025)])
def test_quarter_tile_scores_give_the_sums_of_whole_tiles(kw, lens):
    """A small launch that scores and selects in one call cuts its tiles in four; scored and selected by
    two calls it walks whole tiles.  The statistics, and so the selection scores, are the same bits."""
    w = small(seq_lens=lens, budget=1, window_size=0, **kw)
    inp = build_inputs(w)
    caches, kv, batch, sc = device_objects(w, inp, DEV)
    sel = ops.SelectConfig(window_size=0, allow_resident=False)
    print(f"quarter tiles {kw} {lens}", flush=True)
    keep_a, fin_a, _ = ops.select_paged(kv, batch, sc, sel, want_scores=True)
    raw, ws = ops.score_paged(kv, batch, sc)
    keep_b, fin_b = ops.select(kv, batch, sc, sel, raw, ws, want_scores=True)
    h = w.num_kv_heads
    assert torch.equal(keep_a, keep_b)
    for b, t in enumerate(lens):
        assert torch.equal(fin_a[b * h:(b + 1) * h, :t], fin_b[b * h:(b + 1) * h, :t]), (b, t)


@pytest.mark.parametrize("offsets", [16, 17, 18, 21, 25, 32])
@pytest.mark.parametrize("lens,layers,heads", [((1500, 1, 513), 1, (6, 2)), ((3000, 130, 2049, 511), 16, (40, 8)),
                                               ((2600, 90, 513, 1537), 11, (35, 5)), ((700, 1100), 9, (80, 80))],
                         ids=["a_tile_a_workgroup", "runs_over_units_and_sequences", "runs_not_a_multiple_of_eight", "few_runs_a_head"])
def test_max_aggregation_runs_of_tiles(lens, layers, heads, offsets, monkeypatch):
    """The matrix-core kernel for max aggregation cuts a head's tiles of a ragged batch into equal runs, up to 512 over
    all heads, which end and begin inside layers and sequences, and lays offset 16 out by pieces when it is the only one beyond the
    first sixteen: raw scores against the vector-unit kernel to 1e-5 of the per-head RMS."""
    w = small(num_q_heads=heads[0], num_kv_heads=heads[1], num_layers=layers, seq_lens=lens, budget=64, index=93)
    inp = build_inputs(w)
    print(f"max runs {offsets} {w}", flush=True)
    out = {}
    for kernel in ("mfma", "valu"):
        tune(max_kernel=kernel)
        caches, kv, batch, sc = device_objects(w, inp, DEV, aggregation="max")
        sc = ops.ScoreConfig(sc.folded, sc.omega, torch.arange(offsets, device=DEV, dtype=torch.float32) * 37.0 + 1.0, "max")
        raw, ws = ops.score_paged(kv, batch, sc)
        keep, fin = ops.select(kv, batch, sc, ops.SelectConfig(window_size=0), raw, ws, want_scores=True)
        torch.cuda.synchronize()
        out[kernel] = (raw.clone(), fin.clone())
    h = w.num_kv_heads
    for b, t in enumerate(lens):
        got, want = out["mfma"][0][b, :, :t], out["valu"][0][b, :, :t]
        rms = want.pow(2).mean(dim=1, keepdim=True).sqrt().clamp_min(1e-30)
        assert float(((got - want).abs() / rms).max()) <= 1e-5, b
        fm, fv = out["mfma"][1][b * h:(b + 1) * h, :t], out["valu"][1][b * h:(b + 1) * h, :t]
        assert float((fm - fv).abs().max()) <= SELECT_SCORE_TOL * max(float(fv.abs().max()), 1e-30), b


@pytest.mark.parametrize("lens", [(1,), (15, 128, 129), (2049,), (4096,), (4097, 16)])
@pytest.mark.parametrize("kv_dtype,head_dim,heads,layers,rope", [
    ("bf16", 128, (32, 8), 1, "half"), ("bf16", 128, (12, 4), 3, "interleaved"), ("fp16", 128, (8, 8), 4, "half"),
    ("bf16", 64, (24, 3), 2, "half"), ("fp16", 64, (10, 5), 1, "interleaved"), ("bf16", 256, (4, 2), 2, "interleaved"),
    ("fp16", 256, (14, 2), 1, "half")])
def test_small_launches_match_the_two_pass_kernels(kv_dtype, head_dim, heads, layers, rope, lens, monkeypatch):
    """A few layers of a few requests go through kernels of their own (a wave per step, statistics in the selection's
    workgroups): selection scores and kept sets against the score-then-select kernels, and without
    normalisation, where the raw scores show, to 5e-6 of the largest (two fp32 evaluations of one sum).  The longest
    batch is too much for some shapes, which then take the resident or the two-pass kernels."""
    w = small(kv_dtype=kv_dtype, head_dim=head_dim, num_q_heads=heads[0], num_kv_heads=heads[1], num_layers=layers, rope_style=rope,
              seq_lens=lens, budget=96, index=91)
    print(f"small {w}", flush=True)
    inp = build_inputs(w)
    caches, kv, batch, sc = device_objects(w, inp, DEV, prefill_lens=[5] * len(lens))
    h = w.num_kv_heads
    for kw in (dict(), dict(normalize=False, layer_reduce="max"), dict(group_reduce="mean", protect_prefill=True)):
        sel = ops.SelectConfig(window_size=w.window_size, **kw)
        tune(resident_kernel="auto")
        too_much = lens == (4097, 16) and heads in ((8, 8), (24, 3), (14, 2), (12, 4))
        assert ops.describe_plan(kv, batch, sc, sel)["small_launches"] == (0 if too_much else 1)
        keep_s, fin_s, ws = ops.select_paged(kv, batch, sc, sel, want_scores=True)
        keep_only, _, _ = ops.select_paged(kv, batch, sc, sel)
        tune(resident_kernel="off")
        raw, ws2 = ops.score_paged(kv, batch, sc)
        keep_t, fin_t = ops.select(kv, batch, sc, sel, raw, ws2, want_scores=True)
        torch.cuda.synchronize()
        assert ws.status() == 0
        for b, t in enumerate(lens):
            k = min(w.budget, t)
            assert torch.equal(keep_only[b * h:(b + 1) * h, :k], keep_s[b * h:(b + 1) * h, :k])
            a, c = fin_s[b * h:(b + 1) * h, :t].cpu(), fin_t[b * h:(b + 1) * h, :t].cpu()
            assert torch.equal(torch.isinf(a), torch.isinf(c))
            m = torch.isfinite(c)
            scale = float(c[m].abs().max()) if bool(m.any()) else 1.0
            tol = selection_score_tol(raw[b, :, :t].transpose(-1, -2).cpu()) if sel.normalize else 5e-6
            assert float((a[m] - c[m]).abs().max() if bool(m.any()) else 0.0) <= tol * scale, (kw, b)
            assert_keep_matches(keep_s[b * h:(b + 1) * h, :k].cpu().long(), keep_t[b * h:(b + 1) * h, :k].cpu().long(), c, k,
                                tie_tol=2 * tol * scale)


@pytest.mark.parametrize("kv_dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 6e4])
def test_small_launches_carry_values_beyond_range_like_the_two_pass_kernels(kv_dtype, value, monkeypatch):
    """One key element that is not finite, or as large as its type allows in magnitudes beyond half precision: the raw
    scores keep their kind (finite, infinity and its sign, NaN) and no status is raised."""
    w = small(kv_dtype=kv_dtype, num_q_heads=8, num_kv_heads=2, num_layers=1, seq_lens=(300,), budget=64, window_size=0, index=92)
    inp = build_inputs(w)
    for c in inp["caches"]:
        c[0, inp["tables"][0][3], 5, 1, 7] = value
    caches, kv, batch, sc = device_objects(w, inp, DEV)
    sel = ops.SelectConfig(window_size=0, normalize=False)
    print(f"beyond range {kv_dtype} {value}", flush=True)
    assert ops.describe_plan(kv, batch, sc, sel)["small_launches"] == 1
    _, a, ws = ops.select_paged(kv, batch, sc, sel, want_scores=True)
    tune(resident_kernel="off")
    raw, ws2 = ops.score_paged(kv, batch, sc)
    _, c = ops.select(kv, batch, sc, sel, raw, ws2, want_scores=True)
    torch.cuda.synchronize()
    assert ws.status() == 0
    a, c = a[:, :300].cpu(), c[:, :300].cpu()
    assert torch.equal(torch.isnan(a), torch.isnan(c)) and torch.equal(torch.isinf(a), torch.isinf(c))
    inf = torch.isinf(c)
    assert torch.equal(a[inf], c[inf])
    m = torch.isfinite(c)
    assert float(((a[m] - c[m]).abs() / c[m].abs().clamp_min(1.0)).max()) <= 2e-5


@pytest.mark.parametrize("g", [1, 2, 3, 4, 7, 8])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), float("-inf")])
@pytest.mark.parametrize("layers", [1, 2])
def test_small_launches_rank_values_that_are_no_numbers_like_the_two_pass_kernels(layers, value, g, monkeypatch):
    """One key element that is a NaN or an infinity, with and without normalisation (where it reaches every token of its
    row through the mean), with a guarded window and prefill: the small launches keep what the score-then-select
    kernels keep, token for token where the row holds no finite score, and their scores are of the same kind."""
    w = small(num_q_heads=2 * g, num_kv_heads=2, num_layers=layers, seq_lens=(300,), budget=64, index=94)
    inp = build_inputs(w)
    inp["caches"][0][0, inp["tables"][0][3], 5, 1, 7] = value
    caches, kv, batch, sc = device_objects(w, inp, DEV, prefill_lens=[5])
    print(f"not a number {value} {w}", flush=True)
    for kw in (dict(), dict(normalize=False), dict(group_reduce="mean"), dict(normalize="population"),
               dict(normalize=False, layer_reduce="max", group_reduce="mean")):
        sel = ops.SelectConfig(window_size=w.window_size, protect_prefill=True, **kw)
        tune(resident_kernel="auto")
        assert ops.describe_plan(kv, batch, sc, sel)["small_launches"] == 1
        keep_s, fin_s, ws = ops.select_paged(kv, batch, sc, sel, want_scores=True)
        tune(resident_kernel="off")
        raw, ws2 = ops.score_paged(kv, batch, sc)
        keep_t, fin_t = ops.select(kv, batch, sc, sel, raw, ws2, want_scores=True)
        torch.cuda.synchronize()
        assert ws.status() == 0
        for h in range(2):
            a, c = fin_s[h, :300].cpu(), fin_t[h, :300].cpu()
            got, want = keep_s[h:h + 1, :64].cpu().long(), keep_t[h:h + 1, :64].cpu().long()
            assert torch.equal(torch.isnan(a), torch.isnan(c)) and torch.equal(torch.isinf(a), torch.isinf(c)), (kw, h)
            inf, m = torch.isinf(c), torch.isfinite(c)
            assert torch.equal(a[inf], c[inf]), (kw, h)
            if bool(m.any()):
                scale = float(c[m].abs().max())
                finite = raw[0, :, :300].transpose(-1, -2).cpu()[:, h * g:(h + 1) * g]
                tol = selection_score_tol(finite[torch.isfinite(finite).all(-1).all(-1)]) if sel.normalize else 5e-6
                assert float((a[m] - c[m]).abs().max()) <= tol * scale, (kw, h)
                assert_keep_matches(got, want, c.clone().masked_fill_(torch.isnan(c), float("inf"))[None], 64,
                                    tie_tol=2 * tol * scale)
            else:
                assert torch.equal(got, want), (kw, h, a, c)


@pytest.mark.parametrize("kv_dtype,head_dim,g", [("fp16", 128, 4), ("fp16", 64, 7), ("fp16", 256, 1), ("bf16", 128, 4)])
@pytest.mark.parametrize("what,factor", [("all", 1e-30), ("all", 1e-25), ("all", 1e-20), ("all", 1e-15), ("all", 1e15), ("all", 1e25),
                                         ("trig", 1e-20), ("trig", 1e15), ("norm", 1e-20), ("norm", 1e15)])
def test_small_launches_take_coefficients_of_any_size(what, factor, kv_dtype, head_dim, g, monkeypatch):
    """Statistics far below and above the range of half precision, in both terms of the score or in one of them: the
    scores agree with the two-pass kernels' fp32 arithmetic to 5e-6 of the largest, as with statistics of ordinary size."""
    w = small(kv_dtype=kv_dtype, head_dim=head_dim, num_q_heads=2 * g, num_kv_heads=2, num_layers=1, seq_lens=(300,),
              budget=64, window_size=0, index=95)
    inp = build_inputs(w)
    caches, kv, batch, sc = device_objects(w, inp, DEV)
    sc.folded[:, :, {"all": slice(0, 3), "trig": slice(0, 2), "norm": slice(2, 3)}[what]] *= factor
    sel = ops.SelectConfig(window_size=0, normalize=False)
    print(f"coefficients {what} x {factor} {w}", flush=True)
    assert ops.describe_plan(kv, batch, sc, sel)["small_launches"] == 1
    _, a, ws = ops.select_paged(kv, batch, sc, sel, want_scores=True)
    tune(resident_kernel="off")
    raw, ws2 = ops.score_paged(kv, batch, sc)
    _, c = ops.select(kv, batch, sc, sel, raw, ws2, want_scores=True)
    torch.cuda.synchronize()
    assert ws.status() == 0
    a, c = a[:, :300].double().cpu(), c[:, :300].double().cpu()
    assert bool(torch.isfinite(c).all())
    assert float((a - c).abs().max()) <= 5e-6 * float(c.abs().max())


def test_fp8_every_code_decodes_like_torch():
    """All 254 finite e4m3 codes through the scorer: with one non-zero coefficient the
    score is code_value * scale * coefficient, which pins the decoder against torch's
    float8_e4m3fn conversion (no reference counterpart: the reference has no fp8 code)."""
    codes = torch.tensor([c for c in range(256) if c & 0x7f != 0x7f], dtype=torch.uint8)     # 254 finite codes
    h, d, bs = 2, 128, 16
    t = codes.numel()
    nb = (t + bs - 1) // bs
    g = torch.Generator().manual_seed(5)
    for style in ("half", "interleaved"):
        k = torch.zeros(nb * bs, h, d, dtype=torch.uint8)
        for pos in (0, 5, 63, 64, 77, 127):                      # element positions carrying the code
            k[:t, :, pos] = codes.unsqueeze(1)
        scales = 0.25 + torch.rand(nb * bs, h, generator=g)
        kf8 = k.view(torch.float8_e4m3fn).view(nb, bs, h, d)
        qc = torch.randn(1, h, d // 2, 2, generator=g)
        qa = qc.pow(2).sum(-1).sqrt() + torch.rand(1, h, d // 2, generator=g)
        fs = torch.ones(1, h, d // 2)
        omega, offs = synth.rope_inv_freq(small()), synth.geometric_offsets()
        kd, sd = kf8.to(DEV), scales.to(DEV)
        kv = ops.PagedKV([kd], None, style, [sd], None)
        batch = ops.StepBatch(DEV, [t], round_start=[900], block_tables=[list(range(nb))])
        sc = ops.ScoreConfig(ops.fold_stats(qc.to(DEV), qa.to(DEV), fs.to(DEV)), omega.to(DEV), offs.to(DEV))
        raw, _ = ops.score_paged(kv, batch, sc, head_major=True)
        torch.cuda.synchronize()
        keys = osc.dequant_fp8(kf8.view(nb * bs, h, d), scales)[:t].permute(1, 0, 2)          # [H, T, D]
        want = osc.raw_scores(keys, qc[0], qa[0], omega, offs, fs[0], 900, rope_style=style)
        got = raw[0, 0, :, :t].cpu()
        assert bool(((got - want).abs() <= score_tolerance(want)).all()), style


def test_fp8_step_scores_selects_and_compacts():
    """fp8 cache end to end: kept set against the oracle on dequantised keys, then codes
    and scales of K and V compacted bit-exactly."""
    w = small(kv_dtype="fp8", seq_lens=(700, 150, 60), num_layers=3, num_q_heads=16, num_kv_heads=4, budget=128)
    inp = build_inputs(w)
    caches, kv, batch, sc = device_objects(w, inp, DEV)
    sel = ops.SelectConfig(window_size=w.window_size)
    keep, _ = ops.compress_step(kv, batch, sc, sel)
    torch.cuda.synchronize()
    got = keep.cpu().long()
    h = w.num_kv_heads
    ks_dev, vs_dev = kv._keep[2], kv._keep[3]
    for b, t in enumerate(w.seq_lens):
        k = min(w.budget, t)
        rows = got[b * h:(b + 1) * h, :k]
        if t > w.budget:
            oraw = oracle_raw(w, inp, b, t)
            want, ofin = osel.group_keep_per_head(oraw, h, k, window_size=w.window_size,
                                                  chunk_tokens=osel.score_chunk_tokens(w.block_size, t))
            scale = float(ofin[torch.isfinite(ofin)].abs().max())
            assert assert_keep_matches(rows, want, ofin, k, tie_tol=KEEP_TIE_TOL * scale) == 0
        else:
            assert torch.equal(rows, torch.arange(t).expand(h, t))
    for l in range(w.num_layers):
        ref = inp["caches"][l].clone().view(torch.uint8)
        nb = ref.shape[1]
        ref_s = torch.stack([inp["k_scales"][l].view(nb, w.block_size, h, 1),
                             inp["v_scales"][l].view(nb, w.block_size, h, 1)]).clone()
        dev_c = caches[l].cpu().view(torch.uint8)
        dev_s = torch.stack([ks_dev[l].cpu().view(nb, w.block_size, h, 1), vs_dev[l].cpu().view(nb, w.block_size, h, 1)])
        for b, t in enumerate(w.seq_lens):
            k = min(w.budget, t)
            if k >= t:
                continue
            rows = got[b * h:(b + 1) * h, :k]
            ocp.compact_per_head(ref, inp["tables"][b], w.block_size, rows, t, full_permutation=False)
            ocp.compact_per_head(ref_s, inp["tables"][b], w.block_size, rows, t, full_permutation=False)
            blk, off = ocp.token_slots(inp["tables"][b], w.block_size, torch.arange(k))
            assert torch.equal(dev_c[:, blk, off], ref[:, blk, off]), (l, b)
            assert torch.equal(dev_s[:, blk, off], ref_s[:, blk, off]), (l, b)


@pytest.mark.parametrize("shared", [False, True])
def test_fp8_compaction_moves_scales_with_the_rows(shared):
    """Random keep lists on an fp8 cache with three KV heads and a budget of several scale
    tiles: codes and per-(token, head) scales of K and V bit-exact against the oracle."""
    w = small(kv_dtype="fp8", seq_lens=(3000, 900, 1501), num_layers=2, num_q_heads=3, num_kv_heads=3, budget=1500)
    inp = build_inputs(w)
    caches, kv, batch, _ = device_objects(w, inp, DEV)
    h = w.num_kv_heads
    rows_per = 1 if shared else h
    g = torch.Generator().manual_seed(17)
    keep = torch.zeros(w.num_seqs * rows_per, batch.max_budget, dtype=torch.int32)
    for b, t in enumerate(w.seq_lens):
        k = min(w.budget, t)
        for r in range(rows_per):
            keep[b * rows_per + r, :k] = torch.sort(torch.randperm(t, generator=g)[:k]).values.int()
    print(f"fp8 compaction shared={shared}", flush=True)
    ops.compact(kv, batch, keep.to(DEV), shared=shared)
    torch.cuda.synchronize()
    ks_dev, vs_dev = kv._keep[2], kv._keep[3]
    for l in range(w.num_layers):
        ref = inp["caches"][l].clone().view(torch.uint8)
        nb = ref.shape[1]
        ref_s = torch.stack([inp["k_scales"][l].view(nb, w.block_size, h, 1),
                             inp["v_scales"][l].view(nb, w.block_size, h, 1)]).clone()
        dev_c = caches[l].cpu().view(torch.uint8)
        dev_s = torch.stack([ks_dev[l].cpu().view(nb, w.block_size, h, 1), vs_dev[l].cpu().view(nb, w.block_size, h, 1)])
        for b, t in enumerate(w.seq_lens):
            k = min(w.budget, t)
            rows = keep[b * rows_per:(b + 1) * rows_per, :k].long()
            for tgt in (ref, ref_s):
                if shared:
                    ocp.compact_shared(tgt, inp["tables"][b], w.block_size, rows[0], t, full_permutation=False)
                else:
                    ocp.compact_per_head(tgt, inp["tables"][b], w.block_size, rows, t, full_permutation=False)
            blk, off = ocp.token_slots(inp["tables"][b], w.block_size, torch.arange(k))
            assert torch.equal(dev_c[:, blk, off], ref[:, blk, off]), (l, b)
            assert torch.equal(dev_s[:, blk, off], ref_s[:, blk, off]), (l, b)


def test_fp8_cache_without_row_scales(monkeypatch):
    """A cache with one scale per tensor (vLLM's fp8 KV cache; the codes sit in uint8 tensors):
    the codes are scored as they are and compaction moves rows only.  Selection identical to the
    one with explicit arrays of ones (that path is pinned against the oracle by the fp8 cases
    above), on the two-pass kernels and on the resident one; kept rows bit-exact against the
    oracle's compaction."""
    w = small(kv_dtype="fp8", seq_lens=(300, 45, 1000), num_layers=2)
    inp = build_inputs(w)
    ones = [torch.ones_like(t) for t in inp["k_scales"]]
    caches_a, kv_a, batch, sc = device_objects(w, dict(inp, k_scales=ones, v_scales=ones), DEV)
    caches_b = [c.to(DEV).view(torch.uint8) for c in inp["caches"]]
    kv_b = ops.PagedKV.from_kv_caches(caches_b, w.rope_style)
    assert kv_b.struct.v_scale_layers is None or not kv_b.struct.v_scale_layers
    sel = ops.SelectConfig(window_size=w.window_size)
    for kernel in ("off", "mfma"):
        tune(resident_kernel=kernel)
        print(f"unscaled fp8, resident kernel setting {kernel}", flush=True)
        keep_a, fin_a, _ = ops.select_paged(kv_a, batch, sc, sel, want_scores=True)
        keep_b, fin_b, _ = ops.select_paged(kv_b, batch, sc, sel, want_scores=True)
        torch.cuda.synchronize()
        for b, t in enumerate(w.seq_lens):          # entries beyond a sequence's own budget / length are not written
            rows, k = slice(b * w.num_kv_heads, (b + 1) * w.num_kv_heads), min(w.budget, t)
            assert torch.equal(keep_a[rows, :k], keep_b[rows, :k]), (kernel, b)
            assert torch.equal(fin_a[rows, :t], fin_b[rows, :t]), (kernel, b)
    ops.compact(kv_b, batch, keep_b)
    torch.cuda.synchronize()
    h = w.num_kv_heads
    keep = keep_b.cpu()
    for l in range(w.num_layers):
        ref = inp["caches"][l].clone().view(torch.uint8)
        dev = caches_b[l].cpu()
        for b, t in enumerate(w.seq_lens):
            k = min(w.budget, t)
            ocp.compact_per_head(ref, inp["tables"][b], w.block_size, keep[b * h:(b + 1) * h, :k].long(), t,
                                 full_permutation=False)
            blk, off = ocp.token_slots(inp["tables"][b], w.block_size, torch.arange(k))
            assert torch.equal(dev[:, blk, off], ref[:, blk, off]), (l, b)


def test_invalid_arguments_raise():
    w = small()
    inp = build_inputs(w)
    caches, kv, batch, sc = device_objects(w, inp, DEV)
    with pytest.raises(IndexError):
        bad = ops.StepBatch(DEV, [5000], budgets=96, block_tables=inp["tables"])
        ops.score_paged(kv, bad, sc)
    with pytest.raises(ValueError):
        ops.compact(kv, batch, torch.zeros(3, 5, dtype=torch.int32, device=DEV))
    with pytest.raises(RuntimeError):
        ops.PagedKV.from_kv_caches([c.cpu() for c in caches])


@pytest.mark.parametrize("kernel", ["auto", "mfma", "valu"])
@pytest.mark.parametrize("hq,hkv,decode_start,keep_count", [(8, 2, 40, 96), (14, 2, 0, 64), (4, 4, 17, 200), (8, 2, 290, 50)])
def test_research_path_selection_matches_oracle(hq, hkv, decode_start, keep_count, kernel):
    """``hf_selection.select_keep_indices_per_head`` (decode tokens only, population std clamped at 1e-6,
    group max, layer mean, no window) against ``oracle.selection.hf_keep_per_head``, whose selection is
    pinned by the reference's own ``_select_per_head_independent`` (tests/golden/hf_select.pt); on the
    kernels the library picks for so small a step (the two short launches with up to four query heads, else the
    resident kernel by layers) and on either resident kernel, which evaluate the same population statistics in their gather."""
    from triattention_amd import hf_selection
    if kernel == "valu" and hq // hkv > 4:
        pytest.skip("the vector-unit resident kernel takes up to four query heads per KV head")
    tune(resident_kernel=kernel)
    w = small(num_layers=3, num_q_heads=hq, num_kv_heads=hkv, seq_lens=(300,), budget=keep_count, window_size=0,
              index=80 + hq)
    inp = build_inputs(w)
    t = 300
    kc = [ocp.split_kv(c, inp["kv_axis"])[0] for c in inp["caches"]]
    dense = [ocp.gather_dense(k, inp["tables"][0], w.block_size, 0, t).to(DEV) for k in kc]         # [1, Hkv, T, D]
    folded = ops.fold_stats(inp["qc"].to(DEV), inp["qa"].to(DEV), inp["fs"].to(DEV))
    got = hf_selection.select_keep_indices_per_head(dense, decode_start=decode_start, keep_count=keep_count,
                                                    folded_stats=folded, inv_freq=inp["omega"].to(DEV),
                                                    offsets=inp["offsets"].to(DEV), round_start=t)
    if kernel != "auto" and min(keep_count, t - decode_start) > 0:
        # the step really went to the kernel asked for (the same objects hf_selection builds)
        views = [ks[..., decode_start:, :].permute(0, 2, 1, 3) for ks in dense]
        path = ops.select_path(ops.PagedKV(views, None, "half"),
                               ops.StepBatch(DEV, [t - decode_start], round_start=[t], budgets=[min(keep_count, t - decode_start)]),
                               ops.ScoreConfig(folded, inp["omega"].to(DEV), inp["offsets"].to(DEV), "mean"),
                               ops.SelectConfig(normalize="population", window_size=0, group_reduce="max", layer_reduce="mean"))
        assert path == {"mfma": "resident_mfma", "valu": "resident_valu"}[kernel], path
    oraw = oracle_raw(w, inp, 0, t)
    want, fin = osel.hf_keep_per_head(oraw, hkv, decode_start, keep_count)
    got = got.cpu()
    k = min(keep_count, t - decode_start)
    assert got.dtype == torch.long and tuple(got.shape) == (hkv, decode_start + k)
    assert torch.equal(got[:, :decode_start], want[:, :decode_start])
    assert bool((got[:, 1:] > got[:, :-1]).all())
    if k == t - decode_start:
        assert torch.equal(got, want)
        return
    scale = float(fin.abs().max())
    swapped = assert_keep_matches(got[:, decode_start:] - decode_start, want[:, decode_start:] - decode_start, fin, k,
                                  tie_tol=KEEP_TIE_TOL * scale)
    record_swaps(f"research_path_vs_oracle:{hq}/{hkv}:{decode_start}:{kernel}", swapped, hkv * k)
    assert swapped == 0


@pytest.mark.parametrize("case", ["half_d128", "interleaved_d64", "half_scaled"])
def test_research_path_scores_match_the_references_own_helpers(case):
    """``hf_selection.score_keys_for_round`` -- the kernels on the cache's rotated keys, nothing un-rotated,
    no position table -- against the scores the reference's research path computes for the same keys
    with its own helpers (fixture written by tests/golden/make_hf_score_golden.py: ``invert_rope`` ->
    ``compute_frequency_statistics_from_means`` -> ``score_keys_for_round``, methods/pruning_utils.py), for
    mean and max over the offsets, with and without the MLR term, half and interleaved pairing, key
    positions that do not start at zero and an attention scale of 1.25.  Tolerance: 1e-3 of a head's
    RMS (the two forms evaluate fp32 phases of up to 65536 rad differently; measured ~1e-4)."""
    from triattention_amd import hf_selection
    gold = load_golden("hf_score.pt")[case]
    k_rot = gold["k_rot"].to(DEV).unsqueeze(0)                                  # [1, Hkv, T, D] bf16, as a cache holds them
    qc = torch.stack([gold["q_mean_real"], gold["q_mean_imag"]], dim=-1)
    worst = 0.0
    for tag, mlr in (("", False), ("_nomlr", True)):
        for agg in ("mean", "max"):
            print(f"research path scores: {case} {agg}{tag}", flush=True)
            got = hf_selection.score_keys_for_round(k_rot, qc, gold["q_abs_mean"], gold["inv_freq"], gold["offsets"],
                                                    gold["freq_scale_sq"], int(gold["round_start"]), aggregation=agg,
                                                    rope_style=gold["style"], attention_scale=float(gold["scale"]),
                                                    disable_mlr=mlr).cpu()
            want = gold[f"scores_{agg}{tag}"]
            assert got.shape == want.shape and got.dtype == torch.float32
            rms = want.pow(2).mean(dim=-1, keepdim=True).sqrt()
            err = float(((got - want).abs() / rms).max())
            worst = max(worst, err)
            assert err < 1e-3, (case, agg, tag, err)
    print(f"research path scores: {case} worst error {worst:.2e} of a head's RMS", flush=True)
