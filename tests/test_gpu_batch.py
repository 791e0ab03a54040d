"""GPU parity of batched decode: a batch of independent
sequences in lockstep over a paged KV cache must produce, for every sequence,
the token ids the single-sequence path produces for it alone (which equal the
reference CPU path), with logits within the bound.

Bound: max |batch - single| / max |single| <= 1e-4 for logits (the batch runs
its projections as split-K GEMMs on the fp16 matrix cores with a hi/lo split
of the fp32 activations, the single path as GEMVs); token ids exact.
"""
from __future__ import annotations

import numpy as np
import pytest

from conftest import load_golden, rel_err

pytestmark = pytest.mark.gpu


def synth_model(mmr, g, **overrides):
    return mmr.Model.synthetic(mmr.make_config(**{**g["config"], **overrides}), g["seed"], g["std"], g["round_fp16"])


def single_sequence(mmr, m, prompt, last_index, capacity, kv):
    """seq[0 .. last_index] and last-step logits of one sequence decoded alone."""
    st = m.make_state(capacity, kv)
    st.enqueue_prefill(prompt)
    st.enqueue_decode(last_index - len(prompt))
    st.synchronize()
    return st.read_sequence(0, last_index + 1), st.read_logits()


@pytest.mark.parametrize("kv", ["f16", "f32"])
def test_batch_matches_single_sequences(gpu, kv):
    # prompts of different lengths; positions cross 64-token pages and reach
    # more than four attention tiles (two splits per sequence)
    mmr = gpu
    print(f"[case] batch mini kv={kv}", flush=True)
    g = load_golden("mini")
    m = synth_model(mmr, g)
    kvd = mmr.KV_F16 if kv == "f16" else mmr.KV_F32
    rng = np.random.default_rng(11)
    lengths = [70, 5, 130, 33]
    prompts = [[int(t) for t in rng.integers(0, g["config"]["vocab_size"], n)] for n in lengths]
    cap, steps = 320, 170
    bs = m.make_batch_state(len(prompts), cap, kvd)
    bs.prefill(prompts)
    bs.decode(steps)
    bs.synchronize()
    last = max(lengths) + steps
    assert bs.steps == last
    for b, p in enumerate(prompts):
        ref_seq, ref_logits = single_sequence(mmr, m, p, last, cap, kvd)
        got = bs.read_sequence(b, 0, last + 1)
        np.testing.assert_array_equal(got, ref_seq, err_msg=f"sequence {b}")
        assert rel_err(bs.read_logits(b), ref_logits) < 1e-4, b


def test_batch_wide_hidden_takes_eight_qkv_partials(gpu):
    # hidden 1024: no chunk of up to 256 columns tiles K in three, so the QKV
    # projection hands the attention eight split-K partials (the prologue's
    # full variant; MiniMind2 and the mini model take the three-part one)
    mmr = gpu
    print("[case] batch hidden 1024, 16/2 heads of 64, 8 QKV partials", flush=True)
    g = load_golden("mini")
    m = synth_model(mmr, g, hidden_size=1024, num_attention_heads=16, num_key_value_heads=2, head_dim=64,
                    intermediate_size=1024)
    rng = np.random.default_rng(3)
    lengths = [40, 9, 75]
    prompts = [[int(t) for t in rng.integers(0, g["config"]["vocab_size"], n)] for n in lengths]
    cap, steps = 200, 90
    bs = m.make_batch_state(len(prompts), cap, mmr.KV_F16)
    bs.prefill(prompts)
    bs.decode(steps)
    bs.synchronize()
    last = max(lengths) + steps
    for b, p in enumerate(prompts):
        ref_seq, ref_logits = single_sequence(mmr, m, p, last, cap, mmr.KV_F16)
        np.testing.assert_array_equal(bs.read_sequence(b, 0, last + 1), ref_seq, err_msg=f"sequence {b}")
        assert rel_err(bs.read_logits(b), ref_logits) < 1e-4, b


def test_batch_long_context_split_paths(gpu):
    # positions up to 1150: the attention split count per sequence steps
    # through 1, 2, 4, 8 and 16, so the O projection's staging merges 1-4 and
    # 5-8 split partials itself and hands 16 to the combine kernel
    mmr = gpu
    print("[case] batch mini long context", flush=True)
    g = load_golden("mini")
    m = synth_model(mmr, g)
    rng = np.random.default_rng(5)
    lengths = [20, 3]
    prompts = [[int(t) for t in rng.integers(0, g["config"]["vocab_size"], n)] for n in lengths]
    cap, steps = 1200, 1130
    bs = m.make_batch_state(len(prompts), cap, mmr.KV_F16)
    bs.prefill(prompts)
    bs.decode(steps)
    bs.synchronize()
    last = max(lengths) + steps
    for b, p in enumerate(prompts):
        ref_seq, ref_logits = single_sequence(mmr, m, p, last, cap, mmr.KV_F16)
        np.testing.assert_array_equal(bs.read_sequence(b, 0, last + 1), ref_seq, err_msg=f"sequence {b}")
        assert rel_err(bs.read_logits(b), ref_logits) < 1e-4, b


@pytest.mark.parametrize("batch", [17, 40])
def test_batch_sizes_across_gemm_paths(gpu, batch):
    # 17 rows: the split-K GEMMs' second 16-row tile is partly filled; 40 rows
    # (over 32): the projections fall back to the dense GEMM, whose single
    # "partial" the consumers add, with the separate combine and SwiGLU kernels
    mmr = gpu
    print(f"[case] batch mini B={batch}", flush=True)
    g = load_golden("mini")
    m = synth_model(mmr, g)
    rng = np.random.default_rng(batch)
    lengths = [int(n) for n in rng.integers(1, 40, batch)]
    prompts = [[int(t) for t in rng.integers(0, g["config"]["vocab_size"], n)] for n in lengths]
    cap, steps = 96, 50
    bs = m.make_batch_state(batch, cap, mmr.KV_F16)
    bs.prefill(prompts)
    bs.decode(steps)
    bs.synchronize()
    last = max(lengths) + steps
    for b in (0, batch // 2, batch - 1):
        ref_seq, ref_logits = single_sequence(mmr, m, prompts[b], last, cap, mmr.KV_F16)
        np.testing.assert_array_equal(bs.read_sequence(b, 0, last + 1), ref_seq, err_msg=f"sequence {b}")
        assert rel_err(bs.read_logits(b), ref_logits) < 1e-4, b


@pytest.mark.parametrize("batch,low,high,kv", [(2, 5, 5, "f32"), (2, 700, 720, "f16"), (33, 126, 150, "f16"),
                                               (300, 30, 33, "f32")])
def test_batch_prompt_rows_match_tokenwise(gpu, monkeypatch, batch, low, high, kv):
    # the prompts through the prefill layers against the same prompts through
    # the steps (MMR_PREFILL_TOKENWISE): the fewest rows that take them (4);
    # 699 rows of two sequences; 33 and 300 sequences, whose rows run in two and
    # three passes (4,096 rows over the batch a pass), the last of them ragged
    mmr = gpu
    print(f"[case] batch prompt rows B={batch} {low}..{high} kv={kv}", flush=True)
    g = load_golden("mini")
    m = synth_model(mmr, g)
    kvd = mmr.KV_F16 if kv == "f16" else mmr.KV_F32
    rng = np.random.default_rng(batch + low)
    lengths = [low] + [int(n) for n in rng.integers(low, high + 1, batch - 1)]
    prompts = [[int(t) for t in rng.integers(0, g["config"]["vocab_size"], n)] for n in lengths]
    steps = 6
    last = max(lengths) + steps
    monkeypatch.setenv("MMR_PREFILL_TOKENWISE", "1")
    tok = m.make_batch_state(batch, last, kvd)
    monkeypatch.delenv("MMR_PREFILL_TOKENWISE")
    rows = m.make_batch_state(batch, last, kvd)
    for st in (tok, rows):
        st.prefill(prompts)
        assert st.steps == max(lengths)
        st.decode(steps)
        st.synchronize()
    for b in sorted({0, 1, batch // 2, batch - 1}):
        np.testing.assert_array_equal(rows.read_sequence(b, 0, last + 1), tok.read_sequence(b, 0, last + 1))
        assert rel_err(rows.read_logits(b), tok.read_logits(b)) < 1e-4, b


@pytest.mark.parametrize("d,kv,batch,low,high", [(64, "f32", 64, 101, 110), (96, "f32", 64, 101, 110),
                                                 (64, "f16", 16, 501, 510), (96, "f16", 64, 101, 110)])
def test_batch_prompt_rows_take_many_rows_attention(gpu, monkeypatch, d, kv, batch, low, high):
    # 8 query heads on 2: the 32-query attention kernels over a batch's pages, in
    # two passes of the prompts (the second after cached rows), a last query
    # tile that is not full; against the prompts through the steps
    mmr = gpu
    print(f"[case] batch many-rows attention B={batch} {low}..{high} d={d} kv={kv}", flush=True)
    kvd = mmr.KV_F16 if kv == "f16" else mmr.KV_F32
    cfg = mmr.make_config(hidden_size=8 * d, num_hidden_layers=3, num_attention_heads=8, num_key_value_heads=2,
                          head_dim=d, intermediate_size=512, vocab_size=512, max_position_embeddings=1024,
                          rms_norm_eps=1e-5, rope_theta=1e6, tie_word_embeddings=1)
    m = mmr.Model.synthetic(cfg, 5, 0.02, True)
    passes = -(-(low - 1) * batch // 4096)
    first = mmr.prefill_pass_rows(low - 1, 4096 // batch)
    assert passes == 2 and first % 32 != 0
    for start, tokens in ((0, first), (first, low - 1 - first)):
        assert mmr.prefill_attention_many_rows(8, 2, d, kvd, start, tokens, batch)
    rng = np.random.default_rng(batch + low)
    lengths = [low] + [int(n) for n in rng.integers(low, high + 1, batch - 1)]
    prompts = [[int(t) for t in rng.integers(0, 512, n)] for n in lengths]
    last = max(lengths) + 4
    monkeypatch.setenv("MMR_PREFILL_TOKENWISE", "1")
    tok = m.make_batch_state(batch, last, kvd)
    monkeypatch.delenv("MMR_PREFILL_TOKENWISE")
    rows = m.make_batch_state(batch, last, kvd)
    for st in (tok, rows):
        st.prefill(prompts)
        assert (st.prompt_bytes > 0) is (st is rows)
        st.decode(4)
        st.synchronize()
        assert st.prompt_bytes == 0  # given back
    for b in sorted({0, 1, batch // 2, batch - 1}):
        np.testing.assert_array_equal(rows.read_sequence(b, 0, last + 1), tok.read_sequence(b, 0, last + 1))
        assert rel_err(rows.read_logits(b), tok.read_logits(b)) < (1e-4 if kv == "f32" else 1e-3), b


@pytest.mark.parametrize("switch,value", [("MMR_GEMM_REGISTER_STAGED", "1"), ("MMR_PREFILL_CHUNK", "100")])
def test_batch_prompt_rows_follow_the_switches(gpu, monkeypatch, switch, value):
    # 5 sequences of 61 shared tokens: the other GEMM kernel, and passes of 16
    # tokens of each (80 rows), the last of 13, give the same answer
    mmr = gpu
    print(f"[case] batch prompt rows {switch}={value}", flush=True)
    g = load_golden("mini")
    m = synth_model(mmr, g)
    rng = np.random.default_rng(9)
    prompts = [[int(t) for t in rng.integers(0, g["config"]["vocab_size"], 62 + b)] for b in range(5)]
    plain = m.make_batch_state(5, 80, mmr.KV_F32)
    monkeypatch.setenv(switch, value)
    other = m.make_batch_state(5, 80, mmr.KV_F32)
    for st in (plain, other):
        st.prefill(prompts)
        st.decode(4)
        st.synchronize()
    for b in range(5):
        np.testing.assert_array_equal(other.read_sequence(b, 0, 71), plain.read_sequence(b, 0, 71))
        assert rel_err(other.read_logits(b), plain.read_logits(b)) < 1e-5, b


@pytest.mark.parametrize("megabytes,bitwise", [("0", True), ("1", False)])
def test_batch_prompts_without_the_pass_buffers(gpu, monkeypatch, megabytes, bitwise):
    # no memory for the passes' buffers: the prompts through the steps, bit for
    # bit; 1 MB: shorter passes.  The state answers as ever.
    mmr = gpu
    print(f"[case] batch prompts with {megabytes} MB for passes", flush=True)
    g = load_golden("mini")
    m = synth_model(mmr, g)
    rng = np.random.default_rng(3)
    prompts = [[int(t) for t in rng.integers(0, g["config"]["vocab_size"], 302 + b)] for b in range(9)]
    monkeypatch.setenv("MMR_PREFILL_TOKENWISE", "1")
    tok = m.make_batch_state(9, 320, mmr.KV_F32)
    monkeypatch.delenv("MMR_PREFILL_TOKENWISE")
    monkeypatch.setenv("MMR_PREFILL_BUFFER_MB", megabytes)
    few = m.make_batch_state(9, 320, mmr.KV_F32)
    for st in (tok, few):
        st.prefill(prompts)
        assert st.prompt_bytes <= int(megabytes) << 20
        st.decode(4)
        st.synchronize()
        st.decode(2)
        st.synchronize()
    for b in range(9):
        np.testing.assert_array_equal(few.read_sequence(b, 0, 317), tok.read_sequence(b, 0, 317))
        if bitwise:
            np.testing.assert_array_equal(few.read_logits(b), tok.read_logits(b))
        else:
            assert rel_err(few.read_logits(b), tok.read_logits(b)) < 1e-4, b


def test_batch_reproduces_reference_golden(gpu):
    # MiniMind2 (configs[3] weights): sequence 0 holds the cfg3_short prompt,
    # whose greedy continuation is the reference CPU path's golden output
    mmr = gpu
    g = load_golden("cfg3_short")
    m = synth_model(mmr, g)
    rng = np.random.default_rng(3)
    prompts = [g["prompt"], [int(t) for t in rng.integers(0, 6400, 40)], [int(t) for t in rng.integers(0, 6400, 3)]]
    bs = m.make_batch_state(len(prompts), 128, mmr.KV_F32)
    bs.prefill(prompts)
    bs.decode(len(g["generated"]) - 1 + 40 - len(g["prompt"]))
    got = bs.read_sequence(0, len(g["prompt"]), len(g["generated"])).tolist()
    assert got == g["generated"]
    for b in (1, 2):
        last = bs.steps
        ref_seq, _ = single_sequence(mmr, m, prompts[b], last, 128, mmr.KV_F32)
        np.testing.assert_array_equal(bs.read_sequence(b, 0, last + 1), ref_seq)


def test_batch_graph_replays_match_eager(gpu, monkeypatch):
    mmr = gpu
    g = load_golden("mini")
    m = synth_model(mmr, g)
    prompts = [[1, 2, 3], [4, 5, 6, 7, 8, 9], [10]]
    graph = m.make_batch_state(3, 96)
    monkeypatch.setenv("MMR_NO_GRAPH", "1")
    eager = m.make_batch_state(3, 96)
    monkeypatch.delenv("MMR_NO_GRAPH")
    for st in (graph, eager):
        st.prefill(prompts)
        st.decode(80)
        st.synchronize()
    for b in range(3):
        np.testing.assert_array_equal(graph.read_sequence(b, 0, 87), eager.read_sequence(b, 0, 87))
        np.testing.assert_array_equal(graph.read_logits(b), eager.read_logits(b))


def test_batch_l2_warming_leaves_the_step_unchanged(gpu, monkeypatch):
    # The residual + norm launches' L2-warming blocks (MMR_L2_WARM_BLOCKS; off
    # by default in the batched step) only load the next GEMMs' weights: the
    # batched decode with them equals the decode without, bit for bit, on
    # MiniMind2's shapes (split-K GEMMs for qkv, gate_up, down and lm_head).
    mmr = gpu
    print("[case] batch cfg3 B=8, warming on / off", flush=True)
    g = load_golden("cfg3")
    m = synth_model(mmr, g)
    rng = np.random.default_rng(21)
    prompts = [[int(t) for t in rng.integers(0, g["config"]["vocab_size"], n)] for n in (40, 64, 17, 90, 8, 33, 71, 50)]
    states = []
    for warm in ("128", "0"):
        monkeypatch.setenv("MMR_L2_WARM_BLOCKS", warm)
        bs = m.make_batch_state(len(prompts), 160)
        monkeypatch.delenv("MMR_L2_WARM_BLOCKS")
        bs.prefill(prompts)
        bs.decode(60)
        bs.synchronize()
        states.append(bs)
    last = max(len(p) for p in prompts) + 60
    for b in range(len(prompts)):
        np.testing.assert_array_equal(states[0].read_sequence(b, 0, last + 1), states[1].read_sequence(b, 0, last + 1))
        np.testing.assert_array_equal(states[0].read_logits(b), states[1].read_logits(b))


def test_batch_error_behaviour(gpu):
    mmr = gpu
    g = load_golden("mini")
    m = synth_model(mmr, g)
    V = g["config"]["vocab_size"]
    bs = m.make_batch_state(2, 16)
    with pytest.raises(mmr.InvalidArgument, match="one prompt per sequence"):
        bs.prefill([[1, 2]])
    with pytest.raises(mmr.InvalidArgument, match="cannot be empty"):
        bs.prefill([[1], []])
    with pytest.raises(mmr.OutOfRange):
        bs.prefill([[1], [V]])
    with pytest.raises(mmr.InvalidArgument, match="needs prompts"):
        bs.decode(1)
    with pytest.raises(mmr.LengthError):
        bs.prefill([[1] * 17, [2]])
    bs.prefill([[1, 2, 3], [4]])
    with pytest.raises(mmr.LengthError):
        bs.decode(14)  # 3 + 14 > 16 positions
    bs.decode(13)
    bs.synchronize()
    assert bs.steps == 16
    with pytest.raises(mmr.InvalidArgument, match="empty KV caches"):
        bs.prefill([[1], [2]])
    with pytest.raises(mmr.InvalidArgument):
        m.make_batch_state(0, 16)
    with pytest.raises(mmr.OutOfRange):
        bs.read_sequence(2, 0, 1)
