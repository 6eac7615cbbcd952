"""The one-launch decode step (single sequence): same tokens as the per-stage path and the f64 oracle, logits within
2e-4, across context lengths that change the number of key ranges per head, with the model's options; its bounded
waits give up cleanly when the host makes them."""
import numpy as np
import pytest

from conftest import build_oracle_model, gpu_config

pytestmark = pytest.mark.gpu

TOL_LOGITS = 2e-4


def _quantized(orc, cfg, seed, **kw):
    from async_gpu_amd import workloads
    w = workloads.gpt2_fp32_weights(cfg, seed, std=0.08, **kw)
    return workloads.quantize_gpt2(w, 32, lambda wt, g: orc.quantize_weight_int4(wt, g, orc.SCRIPT))


def _match(got, ref, margins, prompt_len, what):
    n = min(len(got), len(ref))
    diff = [i for i in range(n) if got[i] != ref[i]]
    if diff or len(got) != len(ref):
        i = diff[0] if diff else n
        gap = margins[i - prompt_len] if prompt_len <= i < prompt_len + len(margins) else float("nan")
        pytest.fail(f"{what}: tokens diverge at index {i}; oracle top-1/top-2 gap there {gap:.3e}")


@pytest.mark.parametrize("options", [dict(), dict(gelu=1), dict(argmax_last=1)])
def test_one_launch_equals_per_stage_and_oracle(orc, agpu, dev, options):
    from async_gpu_amd import gpt2, workloads
    cfg = workloads.GPT2_TINY
    qz = _quantized(orc, cfg, 31, nonzero_bias=True, random_ln=True)
    gm = gpt2.Int4Gpt2Model.from_quantized(gpu_config(cfg, **options), qz)
    prompt = workloads.random_prompt(cfg, 8, 7)
    gm.set_decode_mode(gm.DECODE_PER_STAGE)
    (a,), _ = gm.generate_cached(prompt, 40, eos=-1)
    la = gm.last_logits()
    assert not gm.decode_is_one_launch()
    gm.set_decode_mode(gm.DECODE_AUTO)
    (b,), _ = gm.generate_cached(prompt, 40, eos=-1)
    lb = gm.last_logits()
    assert gm.decode_is_one_launch()
    assert np.array_equal(a, b)
    assert np.abs(la - lb).max() <= 1e-5
    (b2,), _ = gm.generate_cached(prompt, 40, eos=-1)
    assert np.array_equal(b, b2) and np.array_equal(lb, gm.last_logits())  # bit-identical run to run
    if not options:
        om = build_oracle_model(cfg, qz)
        ref, margins = om.generate(prompt, 40, cached=True, eos=-1)
        _match(b, ref, margins, 7, "one-launch step")
        om.reset_cache()
        om.forward(ref[:-2], all_rows=False)
        lo = om.forward(ref[-2:-1], all_rows=False)
        assert np.abs(lb[0] - lo[0]).max() <= TOL_LOGITS
    assert gm.decode_floor(8) > 0.0


@pytest.mark.parametrize("d,heads", [(1024, 16), (1280, 20), (1600, 25), (192, 3), (512, 8)])
def test_one_launch_other_model_widths(orc, agpu, dev, d, heads):
    """Widths between the two benchmark models (GPT-2 medium, large, XL) and below them: other tile widths, other numbers
    of tiles per stage (so the stages start at other workgroups and share other ones), tiles above and below the size
    from which a second stage in a row is touched ahead.  Three layers; tokens against the per-stage path and the oracle."""
    from async_gpu_amd import gpt2, workloads
    cfg = dict(n_layer=3, n_embd=d, n_head=heads, vocab=2003, n_positions=96)
    w = workloads.gpt2_fp32_weights(cfg, 5, std=0.05, nonzero_bias=True, random_ln=True)
    qz = workloads.quantize_gpt2(w, 32, lambda wt, g: orc.quantize_weight_int4(wt, g, orc.SCRIPT))
    gm = gpt2.Int4Gpt2Model.from_quantized(gpu_config(cfg), qz)
    prompt = workloads.random_prompt(cfg, 2, 9)
    gm.set_decode_mode(gm.DECODE_PER_STAGE)
    (a,), _ = gm.generate_cached(prompt, 24, eos=-1)
    la = gm.last_logits()
    gm.set_decode_mode(gm.DECODE_AUTO)
    (b,), _ = gm.generate_cached(prompt, 24, eos=-1)
    assert gm.decode_is_one_launch()
    assert np.array_equal(a, b)
    assert np.abs(la - gm.last_logits()).max() <= 2e-5
    om = build_oracle_model(cfg, qz)
    ref, margins = om.generate(prompt, 24, cached=True, eos=-1)
    _match(b, ref, margins, 9, f"one-launch step, d={d}")


@pytest.mark.parametrize("d,heads,group,head,vocab", [(320, 5, 128, "int4", 2003), (192, 3, 64, "f32", 1001), (640, 10, 96, "int4", 515),
                                                      (1280, 20, 128, "f32", 70001), (64, 1, 32, "f32", 63)])
def test_one_launch_other_groups_and_heads(orc, agpu, dev, d, heads, group, head, vocab):
    """Scale groups of more than 32 k (widths that are no multiple of the group, slices of an XCD that begin inside one)
    and the f32 LM head, whose launch follows the step and feeds the token back: against the per-stage path and the
    oracle, in graphs of sixteen steps, a graph of the rest and a single step, and eos-free over several calls."""
    from async_gpu_amd import gpt2, workloads
    cfg = dict(n_layer=2, n_embd=d, n_head=heads, vocab=vocab, n_positions=96)
    w = workloads.gpt2_fp32_weights(cfg, 5, std=0.05, nonzero_bias=True, random_ln=True)
    qz = workloads.quantize_gpt2(w, group, lambda wt, g: orc.quantize_weight_int4(wt, g, orc.SCRIPT), lm_head_int4=head == "int4")
    gm = gpt2.Int4Gpt2Model.from_quantized(
        gpu_config(cfg, group_size=group, lm_head=gpt2.LM_HEAD_INT4 if head == "int4" else gpt2.LM_HEAD_F32, argmax_last=heads == 10), qz)
    prompt = workloads.random_prompt(cfg, 2, 9)
    om = build_oracle_model(cfg, qz, lm_head_int4=head == "int4")
    ref, margins = om.generate(prompt, 36, cached=True, eos=-1)
    gm.set_decode_mode(gm.DECODE_PER_STAGE)
    (a,), _ = gm.generate_cached(prompt, 36, eos=-1)
    la = gm.last_logits()
    gm.set_decode_mode(gm.DECODE_AUTO)
    for n in (36, 2, 36):  # 16 + 16 + 3 steps, one step, and the graphs again
        (b,), _ = gm.generate_cached(prompt, n, eos=-1)
        assert gm.decode_is_one_launch()
        assert np.array_equal(a[:9 + n], b)
        _match(b, ref[:9 + n], margins, 9, f"one-launch step, d={d} group={group} head={head}")
    assert np.abs(la - gm.last_logits()).max() <= 2e-5


@pytest.mark.parametrize("batch,d,heads,group,head,prompt_len", [(2, 128, 2, 32, "int4", 9), (4, 192, 3, 64, "f32", 40), (8, 768, 12, 32, "int4", 20),
                                                                 (3, 1024, 16, 128, "int4", 250), (2, 1600, 25, 32, "int4", 30), (3, 640, 10, 32, "f32", 505),
                                                                 (5, 320, 5, 32, "int4", 254)])
def test_one_launch_for_several_sequences(orc, agpu, dev, batch, d, heads, group, head, prompt_len):
    """Two to eight sequences in one launch per step: four, two and one group of Linear workgroups, head counts that leave
    XCDs without a head, contexts that cross from one key range to two (and, 5 x 320, to where a launch per stage is chosen),
    against the per-stage path; graphs of sixteen steps, of the rest, a single step; the same bits run to run."""
    from async_gpu_amd import gpt2, workloads
    cfg = dict(n_layer=2, n_embd=d, n_head=heads, vocab=512, n_positions=640)
    w = workloads.gpt2_fp32_weights(cfg, 5, std=0.05, nonzero_bias=True, random_ln=True)
    qz = workloads.quantize_gpt2(w, group, lambda wt, g: orc.quantize_weight_int4(wt, g, orc.SCRIPT), lm_head_int4=head == "int4")
    gm = gpt2.Int4Gpt2Model.from_quantized(
        gpu_config(cfg, group_size=group, max_batch=batch + 1, lm_head=gpt2.LM_HEAD_INT4 if head == "int4" else gpt2.LM_HEAD_F32, gelu=batch % 2), qz)
    prompt = np.stack([workloads.random_prompt(cfg, 20 + b, prompt_len) for b in range(batch)])
    gm.set_decode_mode(gm.DECODE_PER_STAGE)
    a, _ = gm.generate_cached(prompt, 36, eos=-1)
    la = gm.last_logits(batch)
    gm.set_decode_mode(gm.DECODE_AUTO)
    before = gm.decode_stats()
    logits = []
    for n in (36, 2, 36):
        b, _ = gm.generate_cached(prompt, n, eos=-1)
        assert all(np.array_equal(x[:prompt_len + n], y) for x, y in zip(a, b))
        logits.append(gm.last_logits(batch))
    assert np.abs(la - logits[0]).max() <= 5e-5 and np.array_equal(logits[0], logits[2])
    one, per_stage = (y - x for x, y in zip(before[:2], gm.decode_stats()[:2]))
    assert one > 0 and one + per_stage == 71 and (per_stage == 0 or batch == 5)
    (c,), _ = gm.generate_cached(prompt[:1], 36, eos=-1)  # one sequence on the same model, then several again
    assert np.array_equal(c, a[0])
    b, _ = gm.generate_cached(prompt[:2], 20, eos=-1)
    assert all(np.array_equal(x[:prompt_len + 20], y) for x, y in zip(a, b))


def test_a_changing_batch_keeps_every_plan(orc, agpu, dev):
    """A caller whose batch changes from call to call: the plans and graphs of every number of sequences stand side by side, so
    once each has been used no device memory is taken or given back any more, and the results stay the same bits."""
    import torch
    from async_gpu_amd import gpt2, workloads
    cfg = dict(n_layer=6, n_embd=768, n_head=12, vocab=512, n_positions=64)
    w = workloads.gpt2_fp32_weights(cfg, 5, std=0.05, nonzero_bias=True, random_ln=True)
    qz = workloads.quantize_gpt2(w, 128, lambda wt, g: orc.quantize_weight_int4(wt, g, orc.SCRIPT))
    gm = gpt2.Int4Gpt2Model.from_quantized(gpu_config(cfg, group_size=128, max_batch=4), qz)
    prompt = np.stack([workloads.random_prompt(cfg, 60 + b, 8) for b in range(4)])

    def run(n):
        toks, _ = gm.generate_cached(prompt[:n], 20, eos=-1)
        return [t.tolist() for t in toks], gm.last_logits(n).copy(), torch.cuda.mem_get_info()[0]

    batches = (4, 1, 3, 2)
    first = {n: run(n) for n in batches}
    for n in (3, 4, 2, 1, 3, 2):
        toks, logits, free = run(n)
        assert toks == first[n][0] and np.array_equal(logits, first[n][1])
        assert free == first[batches[-1]][2]
    assert gm.decode_stats()[1] == 0


@pytest.mark.parametrize("batch", [1, 3])
def test_eager_steps_equal_graph_replays(orc, agpu, dev, batch):
    """The per-stage step launched kernel by kernel gives the bits of its graph replay."""
    from async_gpu_amd import gpt2, workloads
    cfg = workloads.GPT2_TINY
    qz = _quantized(orc, cfg, 33, nonzero_bias=True)
    gm = gpt2.Int4Gpt2Model.from_quantized(gpu_config(cfg, max_batch=4), qz)
    prompt = workloads.random_prompt(cfg, 9, 6, batch=batch)
    gm.set_decode_mode(gm.DECODE_PER_STAGE)
    a, _ = gm.generate_cached(prompt, 30, eos=-1)
    la = gm.last_logits(batch)
    gm.set_decode_mode(gm.DECODE_EAGER)
    b, _ = gm.generate_cached(prompt, 30, eos=-1)
    assert not gm.decode_is_one_launch()
    assert all(np.array_equal(x, y) for x, y in zip(a, b))
    assert np.array_equal(la, gm.last_logits(batch))


@pytest.mark.parametrize("prompt_len", [250, 505, 760])
def test_one_launch_across_key_range_counts(orc, agpu, dev, prompt_len):
    """Beyond 256, 512 and 768 cached positions a head's keys go to two, three and four workgroups."""
    from async_gpu_amd import gpt2, workloads
    cfg = dict(n_layer=2, n_embd=128, n_head=2, vocab=503, n_positions=1024)
    qz = _quantized(orc, cfg, 32, nonzero_bias=True, random_ln=True)
    gm = gpt2.Int4Gpt2Model.from_quantized(gpu_config(cfg), qz)
    om = build_oracle_model(cfg, qz)
    prompt = workloads.random_prompt(cfg, prompt_len, prompt_len)
    ref, margins = om.generate(prompt, 24, cached=True, eos=-1)
    (got,), _ = gm.generate_cached(prompt, 24, eos=-1)
    assert gm.decode_is_one_launch()
    _match(got, ref, margins, prompt_len, f"one-launch step from {prompt_len} positions")
    lb = gm.last_logits()
    gm.set_decode_mode(gm.DECODE_PER_STAGE)
    (per,), _ = gm.generate_cached(prompt, 24, eos=-1)
    assert np.array_equal(per, got)
    assert np.abs(gm.last_logits() - lb).max() <= 1e-5


def test_wait_that_gives_up_is_reported_and_the_model_recovers(orc, agpu, dev):
    """With a limit of two poll rounds every wait inside the step gives up: the kernel still ends, the call reports
    AGPU_ERR_DEVICE_WAIT, and the model serves the same request per stage afterwards."""
    from async_gpu_amd import _lib, gpt2, workloads
    cfg = workloads.GPT2_TINY
    qz = _quantized(orc, cfg, 33)
    gm = gpt2.Int4Gpt2Model.from_quantized(gpu_config(cfg), qz)
    prompt = workloads.random_prompt(cfg, 9, 5)
    (good,), _ = gm.generate_cached(prompt, 12, eos=-1)
    assert gm.decode_is_one_launch()
    gm.set_decode_wait_limit(2)
    with pytest.raises(_lib.AgpuError) as e:
        gm.generate_cached(prompt, 12, eos=-1)
    assert e.value.code == _lib.ERR_DEVICE_WAIT
    assert not gm.decode_is_one_launch()
    (again,), _ = gm.generate_cached(prompt, 12, eos=-1)
    assert not gm.decode_is_one_launch()
    assert np.array_equal(again, good)
    one, per, gave_up, would = gm.decode_stats()
    assert gave_up == 1 and per >= 11 and one >= 11 and not would
    # asked for again (and allowed to wait again), the model plans the one-launch step anew
    gm.set_decode_wait_limit(0)
    gm.set_decode_mode(gm.DECODE_AUTO)
    assert gm.decode_stats()[3]
    (third,), _ = gm.generate_cached(prompt, 12, eos=-1)
    assert gm.decode_is_one_launch()
    assert np.array_equal(third, good)
    assert gm.decode_stats()[2] == 1


@pytest.mark.parametrize("batch,d,heads,group,head", [(3, 128, 2, 32, "int4"), (8, 192, 3, 64, "f32"), (2, 1600, 25, 32, "int4"), (1, 128, 2, 32, "f32"),
                                                      (1, 192, 3, 64, "int4")])
def test_a_wait_that_gives_up_with_several_sequences_other_heads_and_groups(orc, agpu, dev, batch, d, heads, group, head):
    """The same for the other steps that are one launch: several sequences, the f32 head, longer groups.  The step and the launches behind
    it run to their end; generate_cached and the sampling run the request again per stage by themselves (the generator's state
    as well), so their callers get what they would have got; decode_steps, which has no prompt to begin from again, reports."""
    from async_gpu_amd import _lib, gpt2, ops, workloads
    cfg = dict(n_layer=2, n_embd=d, n_head=heads, vocab=503, n_positions=96)
    w = workloads.gpt2_fp32_weights(cfg, 5, std=0.05, nonzero_bias=True, random_ln=True)
    qz = workloads.quantize_gpt2(w, group, lambda wt, g: orc.quantize_weight_int4(wt, g, orc.SCRIPT), lm_head_int4=head == "int4")
    gm = gpt2.Int4Gpt2Model.from_quantized(
        gpu_config(cfg, group_size=group, max_batch=batch, lm_head=gpt2.LM_HEAD_INT4 if head == "int4" else gpt2.LM_HEAD_F32), qz)
    prompt = np.stack([workloads.random_prompt(cfg, 70 + b, 9) for b in range(batch)])
    good, _ = gm.generate_cached(prompt, 24, eos=-1)
    assert gm.decode_stats()[:3] == (23, 0, 0)
    gm.set_decode_wait_limit(2)
    again, _ = gm.generate_cached(prompt, 24, eos=-1)
    assert all(np.array_equal(x, y) for x, y in zip(good, again))
    one, per, gave_up, _ = gm.decode_stats()
    assert one == 46 and per == 23 and gave_up == 1
    gm.set_decode_mode(gm.DECODE_AUTO)
    longer, _ = gm.generate_cached(prompt, 84, eos=-1)  # long enough for the model to look at the one-launch step again meanwhile
    assert all(np.array_equal(x, y[:33]) for x, y in zip(good, longer))
    assert gm.decode_stats()[1:3] == (23 + 83, 2)
    gm.set_decode_mode(gm.DECODE_AUTO)  # asked for again, still with the limit
    gm.reset_cache()
    gm.forward_cached(prompt, all_rows=False)
    with pytest.raises(_lib.AgpuError) as e:
        gm.decode_steps(batch, 5)
    assert e.value.code == _lib.ERR_DEVICE_WAIT and gm.decode_stats()[2] == 3
    if batch == 1:
        gm.set_decode_wait_limit(0)
        gm.set_decode_mode(gm.DECODE_AUTO)
        r0, r1 = ops.SimpleRng(7), ops.SimpleRng(7)
        a = gm.generate_cached_sampling(prompt[0], 20, 5, 0.9, r0, eos=-1)
        assert gm.decode_stats()[2] == 3
        gm.set_decode_wait_limit(2)
        b = gm.generate_cached_sampling(prompt[0], 20, 5, 0.9, r1, eos=-1)
        assert gm.decode_stats()[2] == 4
        assert np.array_equal(a, b) and r0.next_f32() == r1.next_f32()
    gm.set_decode_wait_limit(0)
    gm.set_decode_mode(gm.DECODE_AUTO)
    before = gm.decode_stats()
    third, _ = gm.generate_cached(prompt, 24, eos=-1)
    assert all(np.array_equal(x, y) for x, y in zip(good, third))
    assert gm.decode_stats()[0] == before[0] + 23


def test_a_model_that_fell_back_tries_the_one_launch_step_again_after_a_while(orc, agpu, dev):
    """Without being asked, the model looks at the one-launch step again after 64 looks at the decode path."""
    from async_gpu_amd import _lib, gpt2, workloads
    cfg = workloads.GPT2_TINY
    qz = _quantized(orc, cfg, 35)
    gm = gpt2.Int4Gpt2Model.from_quantized(gpu_config(cfg), qz)
    prompt = workloads.random_prompt(cfg, 11, 5)
    (good,), _ = gm.generate_cached(prompt, 20, eos=-1)
    gm.set_decode_wait_limit(2)
    with pytest.raises(_lib.AgpuError):
        gm.generate_cached(prompt, 20, eos=-1)
    gm.set_decode_wait_limit(0)  # whatever was in the way is gone
    came_back = False
    for _ in range(40):
        (got,), _ = gm.generate_cached(prompt, 20, eos=-1)
        assert np.array_equal(got, good)
        if gm.decode_is_one_launch():
            came_back = True
            break
    assert came_back
    assert gm.decode_stats()[2] == 1


@pytest.mark.parametrize("last", [0, 1])
@pytest.mark.parametrize("mode", ["one_launch", "per_stage"])
def test_f32_head_picks_among_ties_and_nan(orc, agpu, dev, last, mode):
    """The launch that is the f32 head picks the token too: of equal logits the first, or the last with argmax_last; a NaN logit never
    wins; nothing comparable is token 0.  Every row of the embedding has a twin 250 rows on, so every maximum is a tie."""
    from async_gpu_amd import gpt2, workloads
    cfg = dict(n_layer=2, n_embd=192, n_head=3, vocab=503, n_positions=64)
    w = workloads.gpt2_fp32_weights(cfg, 5, std=0.08, nonzero_bias=True, random_ln=True)
    w["wte"][250:500] = w["wte"][:250]
    prompt = np.array([3, 1, 4, 1, 5], np.uint32)

    def step(wte, lnf_g):
        qz = workloads.quantize_gpt2(dict(w, wte=wte, lnf_g=lnf_g), 32, lambda wt, g: orc.quantize_weight_int4(wt, g, orc.SCRIPT), lm_head_int4=False)
        gm = gpt2.Int4Gpt2Model.from_quantized(gpu_config(cfg, lm_head=gpt2.LM_HEAD_F32, argmax_last=last), qz)
        gm.set_decode_mode(gm.DECODE_AUTO if mode == "one_launch" else gm.DECODE_PER_STAGE)
        (t,), _ = gm.generate_cached(prompt, 6, eos=-1)
        assert gm.decode_is_one_launch() == (mode == "one_launch")
        return t, gm.last_logits()[0]

    t, logits = step(w["wte"], w["lnf_g"])
    winners = np.flatnonzero(logits == logits.max())
    assert len(winners) == 2 or winners[0] >= 500
    assert t[-1] == winners[-1 if last else 0]
    assert all((x >= 250) == bool(last) for x in t[len(prompt):] if x < 500)
    wte = w["wte"].copy()  # the winner and its twin out of the way
    wte[winners] = np.nan
    t, logits = step(wte, w["lnf_g"])
    assert np.isnan(logits[winners]).all() and np.isfinite(np.delete(logits, winners)).all()
    left = np.flatnonzero(logits == np.nanmax(logits))
    assert t[-1] == left[-1 if last else 0]
    t, logits = step(w["wte"], np.full_like(w["lnf_g"], np.nan))
    assert np.isnan(logits).all() and all(x == 0 for x in t[len(prompt):])


def test_one_launch_step_on_raw_nibbles_over_the_whole_range(orc, agpu, dev):
    """The Linear inside the one-launch step, pinned on its own: one block of GPT-2 small's width whose packed words are
    drawn directly (nibbles uniform over all sixteen values, so the value -8 that the quantizer never emits is there;
    scales U(0.002, 0.02): BASELINE config 1's distribution, compute_gemm.rs:2882-2895), non-zero biases, random LayerNorm
    gains and offsets, and embedding rows whose magnitudes span four decades.  The logits of every decode step against
    the f64 oracle on the same token sequence (2e-4 of the largest logit magnitude), and against the per-stage path."""
    from async_gpu_amd import gpt2, workloads
    cfg = dict(n_layer=1, n_embd=768, n_head=12, vocab=2003, n_positions=32)
    d, ff, V, P = 768, 3072, cfg["vocab"], cfg["n_positions"]
    rng = np.random.default_rng(77)
    layer = dict(ln1_g=(1.0 + 0.1 * rng.standard_normal(d)).astype(np.float32), ln1_b=(0.1 * rng.standard_normal(d)).astype(np.float32),
                 ln2_g=(1.0 + 0.1 * rng.standard_normal(d)).astype(np.float32), ln2_b=(0.1 * rng.standard_normal(d)).astype(np.float32))
    for name, (k, n) in zip(workloads.LINEAR_NAMES, ((d, 3 * d), (d, d), (d, ff), (ff, d))):
        layer[name] = workloads.random_int4_linear(rng, k, n, 32, bias=True)
    head_packed, head_scales, _ = workloads.random_int4_linear(rng, d, V, 32)
    wte = (rng.standard_normal((V, d)) * 10.0 ** rng.uniform(-2, 2, size=(V, 1))).astype(np.float32)
    wpe = (0.01 * rng.standard_normal((P, d))).astype(np.float32)
    qz = dict(group=32, wte=wte, wpe=wpe, lnf_g=(1.0 + 0.1 * rng.standard_normal(d)).astype(np.float32),
              lnf_b=(0.1 * rng.standard_normal(d)).astype(np.float32), layers=[layer], lm_head=(head_packed, head_scales))
    assert any((layer[n][0] & 0xF == 0).any() for n in workloads.LINEAR_NAMES)  # the nibble of -8 is among the weights
    gm = gpt2.Int4Gpt2Model.from_quantized(gpu_config(cfg), qz)
    om = build_oracle_model(cfg, qz)
    prompt = workloads.random_prompt(cfg, 12, 6)
    for steps in (2, 3, 9):
        gm.set_decode_mode(gm.DECODE_AUTO)
        (got,), _ = gm.generate_cached(prompt, steps, eos=-1)
        assert gm.decode_is_one_launch()
        lg = gm.last_logits()[0]
        om.reset_cache()
        lo = om.forward(got[:-1], all_rows=False)[0]
        scale = max(1.0, float(np.abs(lo).max()))
        err = float(np.abs(lg - lo).max())
        assert err <= TOL_LOGITS * scale, f"{steps - 1} decode steps: logits differ from the oracle's by {err:.3e} (largest logit {scale:.3e})"
        gm.set_decode_mode(gm.DECODE_PER_STAGE)
        (per,), _ = gm.generate_cached(prompt, steps, eos=-1)
        lp = gm.last_logits()[0]
        if np.array_equal(per, got):  # the same sequence (a near tie may part them): the two paths' logits side by side
            assert float(np.abs(lp - lg).max()) <= TOL_LOGITS * scale


@pytest.mark.parametrize("mode", ["one_launch", "per_stage"])
def test_weights_replaced_under_cached_graphs_are_the_ones_the_next_call_uses(orc, agpu, dev, mode):
    """Every setter that can replace a buffer or a folded vector drops the cached graphs and the step's plan: a model
    that has decoded, then gets other LayerNorm vectors, one other Linear and other embeddings, decodes like a model built
    with them from scratch (and like neither of the two it was before)."""
    from async_gpu_amd import gpt2, workloads
    cfg = workloads.GPT2_TINY
    qa = _quantized(orc, cfg, 51, nonzero_bias=True, random_ln=True)
    qb = _quantized(orc, cfg, 52, nonzero_bias=True, random_ln=True)
    prompt = workloads.random_prompt(cfg, 9, 6)

    def run(m):
        m.set_decode_mode(m.DECODE_AUTO if mode == "one_launch" else m.DECODE_PER_STAGE)
        (t,), _ = m.generate_cached(prompt, 24, eos=-1)
        assert m.decode_is_one_launch() == (mode == "one_launch")
        return t, m.last_logits().copy()

    gm = gpt2.Int4Gpt2Model.from_quantized(gpu_config(cfg), qa)
    ta, la = run(gm)
    # a mix: embeddings and LayerNorms of b, Linears of a except layer 1's fc, the head of b
    mix = dict(qa, wte=qb["wte"], wpe=qb["wpe"], lnf_g=qb["lnf_g"], lnf_b=qb["lnf_b"], lm_head=qb["lm_head"])
    mix["layers"] = [dict(L) for L in qa["layers"]]
    for li, L in enumerate(mix["layers"]):
        for k in ("ln1_g", "ln1_b", "ln2_g", "ln2_b"):
            L[k] = qb["layers"][li][k]
    mix["layers"][1]["fc"] = qb["layers"][1]["fc"]
    gm.set_embeddings(mix["wte"], mix["wpe"], mix["lnf_g"], mix["lnf_b"])
    for li, L in enumerate(mix["layers"]):
        gm.set_layer_norms(li, L["ln1_g"], L["ln1_b"], L["ln2_g"], L["ln2_b"])
    gm.set_int4_linear(1, "fc", *mix["layers"][1]["fc"])
    gm.set_int4_linear(-1, 0, mix["lm_head"][0], mix["lm_head"][1], None)
    tm, lm = run(gm)
    fresh = gpt2.Int4Gpt2Model.from_quantized(gpu_config(cfg), mix)
    tf, lf = run(fresh)
    assert np.array_equal(tm, tf) and np.array_equal(lm, lf)
    assert not np.array_equal(la, lm)


def test_sampling_runs_on_the_one_launch_step(orc, agpu, dev):
    from async_gpu_amd import gpt2, ops, workloads
    cfg = workloads.GPT2_TINY
    qz = _quantized(orc, cfg, 34)
    gm = gpt2.Int4Gpt2Model.from_quantized(gpu_config(cfg), qz)
    prompt = workloads.random_prompt(cfg, 10, 6)
    a = gm.generate_cached_sampling(prompt, 20, 5, 0.9, ops.SimpleRng(7), eos=-1)
    assert gm.decode_is_one_launch()
    gm.set_decode_mode(gm.DECODE_PER_STAGE)
    b = gm.generate_cached_sampling(prompt, 20, 5, 0.9, ops.SimpleRng(7), eos=-1)
    assert np.array_equal(a, b)


@pytest.mark.parametrize("batch,d,heads,group,head,offset", [(1, 768, 12, 128, "f32", 0.0), (1, 768, 12, 32, "int4", 3.0), (2, 768, 12, 128, "f32", 0.0),
                                                             (3, 1024, 16, 32, "int4", 3.0), (8, 768, 12, 64, "f32", 3.0)])
def test_one_launch_step_is_as_exact_as_an_explicit_layer_norm(orc, agpu, dev, batch, d, heads, group, head, offset):
    """The step's LayerNorms are folded into the Linears behind them.  That must not cost accuracy: neither where the rows'
    mean is zero nor where it is a multiple of their standard deviation (an offset on every position's embedding).  The
    relative 2-norm error of the last step's logits against the f64 oracle; a Linear sums about 1000 products whose
    additions round at 2^-24 of a partial sum (rms 0.3 x 2^-24 each, some 20 of them in the longest chain): 1e-7 per Linear,
    and the eight or nine Linears of two blocks and the head add up to 3e-7 in rms.  The offset costs what the residual
    stream itself loses by it (its additions round at 3.2 instead of 1 standard deviation): 3.2 x 2^-24 x 0.3 per addition and
    element, 2e-7 more.  Half as much again is allowed: 4.5e-7 and 7.5e-7.  (Measured 3.1e-7 and 3.0 - 3.8e-7; sums over unsigned nibbles and rows with their mean: 5.6e-7 and 1.2 - 1.7e-6.)"""
    from async_gpu_amd import gpt2, workloads
    cfg = dict(n_layer=2, n_embd=d, n_head=heads, vocab=1003, n_positions=64)
    w = workloads.gpt2_fp32_weights(cfg, 11, std=0.02, nonzero_bias=True, random_ln=True)
    w["wpe"] = (w["wpe"] + np.float32(offset * 0.02 * np.sqrt(2.0))).astype(np.float32)
    qz = workloads.quantize_gpt2(w, group, lambda wt, g: orc.quantize_weight_int4(wt, g, orc.SCRIPT), lm_head_int4=head == "int4")
    gm = gpt2.Int4Gpt2Model.from_quantized(
        gpu_config(cfg, group_size=group, max_batch=batch, lm_head=gpt2.LM_HEAD_INT4 if head == "int4" else gpt2.LM_HEAD_F32), qz)
    om = build_oracle_model(cfg, qz, lm_head_int4=head == "int4")
    prompt = np.stack([workloads.random_prompt(cfg, 40 + b, 24) for b in range(batch)])
    toks, _ = gm.generate_cached(prompt, 4, eos=-1)
    assert gm.decode_stats()[0] == 3
    lg = gm.last_logits(batch)
    err = []
    for b in range(batch):
        om.reset_cache()
        lo = om.forward(np.asarray(toks[b][:-1]), all_rows=False)[0]
        err.append(np.sqrt(((lg[b] - lo) ** 2).mean() / (lo ** 2).mean()))
    rms = float(np.sqrt(np.mean(np.square(err))))
    print(f"relative error {rms:.2e}")
    assert rms <= (7.5e-7 if offset else 4.5e-7), f"logits are {rms:.2e} off"
