"""Hybrid decoders (the Lozupel design), the parts that need no GPU: the config reader, the order
of layer runs, the fused weight layout, state-slot bookkeeping in the scheduler, and the float32
restatement's own invariants (a window edge, a state carried across a cut)."""
import numpy as np
import pytest
import torch

from oracle import lozupel_ref as R


def _cfg(loop=None, softcap=9.0):
    left = {"heads": 4, "kv_heads": 2, "dim": 16, "vdim": 24, "mask": {"size": 5}, "rot": {"dims": 8, "base": 100.0},
            "scale": 0.3}
    d = {"architecture": "Lozupel", "embedding": {"scale": 2.0}, "width": 40, "vocab": 50, "norm": {"eps": 1e-5},
         "layers": [{"type": "parallel", "mixer": {"left": left, "right": {"heads": 2, "kv_heads": 1, "dim": 16, "vdim": 8, "conv": 3}},
                     "mlp": {"kind": "dense", "ff": 56}},
                    {"type": "delta", "mixer": {"heads": 2, "kv_heads": 2, "dim": 8, "vdim": 16, "conv": 2}, "mlp": None},
                    {"type": "delta", "mixer": {"heads": 1, "kv_heads": 1, "dim": 8, "vdim": 8, "conv": 4},
                     "mlp": {"kind": "dense", "ff": 24}}]}
    if loop:
        d["loop"] = loop
    if softcap:
        d["logit_softcap"] = softcap
    return d


def test_config_reader_and_layer_runs():
    from mi355_decode.config import ModelConfig
    c = ModelConfig.from_dict(_cfg(loop={"start": 1, "stop": 3, "times": 2}))
    assert c.family == "hybrid" and c.architecture == "Lozupel" and c.hidden_size == 40 and c.vocab_size == 50
    s = c.hybrid
    assert s.embed_scale == 2.0 and s.logit_softcap == 9.0 and c.rms_norm_eps == 1e-5
    assert s.runs() == [(0, None), (1, 0), (2, 0), (1, 1), (2, 1)] == R.layer_runs(_cfg(loop={"start": 1, "stop": 3, "times": 2}))
    a, d = s.layers[0].attn, s.layers[0].delta
    assert (a.heads, a.kv_heads, a.dim, a.vdim, a.window, a.rot_dims, a.rot_base, a.scale) == (4, 2, 16, 24, 5, 8, 100.0, 0.3)
    assert d.per_channel and d.conv == 3 and not s.layers[1].delta.per_channel
    assert s.layers[0].ff == 56 and s.layers[1].ff is None
    plain = ModelConfig.from_dict(_cfg(softcap=None)).hybrid
    assert plain.runs() == [(0, None), (1, None), (2, None)] and plain.logit_softcap is None
    whole = ModelConfig.from_dict(_cfg(loop={"start": 0, "stop": 3, "times": 3})).hybrid
    assert whole.runs() == [(i, t) for t in range(3) for i in range(3)]
    with pytest.raises(ValueError):
        ModelConfig.from_dict(_cfg(loop={"start": 2, "stop": 5, "times": 2}))
    bad = _cfg()
    bad["layers"][1]["type"] = "other"
    with pytest.raises(ValueError):
        ModelConfig.from_dict(bad)


def test_weight_layout_fuses_what_reads_the_layer_input():
    from mi355_decode import weights as W
    from mi355_decode.config import ModelConfig
    cfgd = _cfg(loop={"start": 1, "stop": 2, "times": 2})
    st = R.random_state(cfgd, seed=3, rank=5)
    c = ModelConfig.from_dict(cfgd)
    w = W.from_state_dict(c, st, torch.float32, "cpu")
    lw = w.layers[0]
    for name, key in (("lq", "l0.mix.left.q"), ("lg", "l0.mix.left.g"), ("q", "l0.mix.right.q"), ("b", "l0.mix.right.b"),
                      ("a1", "l0.mix.right.a1"), ("g1", "l0.mix.right.g1")):
        at, n = lw.seg[name]
        assert at % 8 == 0 and torch.equal(lw.in_w[at:at + n], st[key])
    q0 = lw.seg["q"][0]
    assert lw.seg["k"][0] == q0 + 16 and lw.seg["v"][0] == q0 + 32          # adjacent: one convolution launch
    assert torch.equal(lw.conv_w, torch.cat([st["l0.mix.right.q.conv"], st["l0.mix.right.k.conv"], st["l0.mix.right.v.conv"]]))
    assert lw.a2_w.shape == (2 * 16, 5) and lw.dt_bias.shape == (32,) and lw.dt_bias.dtype == torch.float32
    assert torch.equal(lw.gate_up_w, torch.cat([st["l0.mix.mlp.gate"] if False else st["l0.mlp.gate"], st["l0.mlp.up"]]))
    assert w.layers[1].norm2 is None and w.layers[1].gate_up_w is None and w.layers[1].dt_bias.shape == (2,)
    assert w.loop_step.shape == (2, 40) and w.final_norm.shape == (1,)
    del st["l2.mix.a"]
    with pytest.raises(KeyError):
        W.from_state_dict(c, st, torch.float32, "cpu")
    with pytest.raises(ValueError):
        W.from_state_dict(c, R.random_state(cfgd, 3), torch.float32, "cpu", tp_size=2)
    syn = W.hybrid_synthetic_state(c, seed=1, rank=7)
    assert set(syn) == set(R.random_state(cfgd, 0, rank=7)) and syn["l0.mix.right.a2"].shape == (32, 7)


def test_state_slots_follow_a_sequence_through_the_scheduler():
    from mi355_decode.engine import BlockAllocator, NoFreeBlocks, Scheduler, Sequence, SlotAllocator
    from mi355_decode.sampling_params import SamplingParams
    slots = SlotAllocator(2)
    sched = Scheduler(BlockAllocator(8), max_num_seqs=4, max_num_batched_tokens=64, max_model_len=128, slots=slots)
    seqs = [Sequence(str(i), list(range(20)), SamplingParams(max_tokens=4)) for i in range(3)]
    for s in seqs:
        sched.add(s)
    kind, chunks = sched.schedule()
    assert kind == "prefill" and [c[0] for c in chunks] == seqs[:2]            # the third waits for a slot
    assert sorted(s.state_slot for s in seqs[:2]) == [0, 1] and seqs[2].state_slot is None and slots.num_free == 0
    for s, _, n in chunks:
        s.num_computed = n
    freed = seqs[0].state_slot
    sched.release(seqs[0])
    assert seqs[0].state_slot is None and slots.num_free == 1
    kind, chunks = sched.schedule()
    assert kind == "prefill" and chunks[0][0] is seqs[2] and seqs[2].state_slot == freed
    late = Sequence("late", [], SamplingParams(max_tokens=1))
    with pytest.raises(NoFreeBlocks):
        sched.admit(late, 5)
    assert late.state_slot is None and late not in sched.running


def test_restatement_window_edge_and_cut_invariance():
    """The float32 restatement itself: a loud key is heard window - 1 tokens later and not after;
    the delta rule gives the same outputs when the sequence is cut and the state carried by hand."""
    T, d = 12, 4
    q = torch.zeros(T, 1, d)
    q[:, 0, 0] = 6.0
    k = torch.zeros(T, 1, d)
    k[2, 0, 0] = 6.0
    v = torch.zeros(T, 1, 2)
    v[2, 0, 1] = 1.0
    o = R.sigmoid_window_attention(q, k, v, 5, 1.0, torch.ones(1), torch.full((1,), -30.0))
    assert o[6, 0, 1] > 0.99 and o[7, 0, 1] < 1e-9 and o[1, 0, 1] == 0
    g = torch.Generator().manual_seed(0)
    x, w = torch.randn(9, 3, generator=g), torch.randn(3, 4, generator=g)
    y = R.short_conv_silu(x, w)
    assert torch.allclose(y[0], torch.nn.functional.silu(x[0] * w[:, 3]))
    assert torch.allclose(y[5], torch.nn.functional.silu((x[2:6] * w.T).sum(0)))
    cfgd = _cfg(loop={"start": 0, "stop": 2, "times": 2})
    wts = R.random_state(cfgd, 5)
    toks = list(range(30))
    z = R.forward(wts, cfgd, toks)
    assert torch.allclose(R.forward(wts, cfgd, toks[:17]), z[:17], atol=1e-5)     # causal
    assert float(z.abs().max()) <= 9.0


class _StatefulRunner:
    """A runner double whose 'model' is a running checksum per state slot and a token table in the KV
    pages: it fails loudly when a step hands it a slot whose state does not continue the request, a
    page that holds another request's tokens, or a chunk at position 0 that finds old state."""
    device, V, NUM_STAGES = "cpu", 50, 1

    def __init__(self, num_blocks, max_num_seqs, max_model_len, slots):
        import numpy as np
        self.np = np
        self.num_blocks, self.max_num_seqs, self.num_state_slots = num_blocks, max_num_seqs, slots
        self.max_blocks = (max_model_len + 15) // 16
        self.pages = np.full(num_blocks * 16, -1, dtype=np.int64)
        self.state = {s: (0, 0) for s in range(slots)}          # slot -> (tokens seen, checksum)
        self.batches = []

    def host_inputs(self, stage=0):
        B = self.max_num_seqs
        return self.np.zeros(3 * B, dtype=self.np.int64), self.np.zeros(B + B * self.max_blocks + B, dtype=self.np.int32)

    def run_prefill(self, token_ids, positions, slot_mapping, block_tables, cu_seqlens, context_lens, max_q_len,
                    sampling=None, logprobs=-1, prompt_logprobs=None, state_slots=None, logit_rows=None):
        np = self.np
        assert state_slots is not None and len(state_slots) == len(context_lens) and len(set(state_slots.tolist())) == len(state_slots)
        self.batches.append([int(cu_seqlens[i + 1] - cu_seqlens[i]) for i in range(len(context_lens))])
        rows = np.zeros((len(token_ids), self.V), dtype=np.float32)
        for i, slot in enumerate(state_slots.tolist()):
            a, b = int(cu_seqlens[i]), int(cu_seqlens[i + 1])
            start = int(positions[a])
            seen, acc = (0, 0) if start == 0 else self.state[slot]
            assert seen == start, f"slot {slot} holds {seen} tokens, the chunk starts at {start}"
            for r in range(a, b):
                self.pages[slot_mapping[r]] = token_ids[r]
                acc = (acc * 31 + int(token_ids[r]) + 1) % 1000003
                p = int(positions[r])
                ctx = self.pages[block_tables[i][np.arange(p + 1) // 16].astype(np.int64) * 16 + np.arange(p + 1) % 16]
                rows[r, 0], rows[r, 1] = acc, int(ctx.sum())    # what the state and what the pages remember
            self.state[slot] = (start + b - a, acc)
        return rows[np.asarray(logit_rows, dtype=np.int64)]


def test_forced_steps_keep_pages_and_slots_straight():
    """LLMEngine.forced_step on a double: mixed batches, a request that sits out, requests that end
    and hand their pages and slot to newcomers; every wanted row equals what the request alone gives."""
    import numpy as np
    from mi355_decode.engine import LLMEngine
    runner = _StatefulRunner(num_blocks=12, max_num_seqs=3, max_model_len=96, slots=3)
    eng = LLMEngine(runner, max_num_seqs=3, max_num_batched_tokens=1 << 20, max_model_len=96)
    rng = np.random.default_rng(0)
    toks = {r: rng.integers(0, 50, n).tolist() for r, n in (("a", 40), ("b", 17), ("c", 5), ("d", 33), ("e", 64))}

    def alone(t):
        acc, out = 0, []
        for i, x in enumerate(t):
            acc = (acc * 31 + x + 1) % 1000003
            out.append((acc, sum(t[: i + 1])))
        return out

    plan = [([("a", 16), ("b", 2), ("c", 5)], ["c"]), ([("a", 1), ("d", 20)], []), ([("a", 23), ("b", 15), ("d", 1)], ["a", "b"]),
            ([("d", 12), ("e", 64)], ["d", "e"])]
    at = {r: 0 for r in toks}
    for entries, end in plan:
        req = [(r, toks[r][at[r]:at[r] + n], [0, n - 1] if n > 1 else [0]) for r, n in entries]
        out = eng.forced_step(req, end)
        row = 0
        for r, t, want in req:
            for j in want:
                assert tuple(out[row][:2]) == tuple(float(v) for v in alone(toks[r])[at[r] + j]), (r, j)
                row += 1
            at[r] += len(t)
        assert row == out.shape[0]
    assert all(at[r] == len(toks[r]) for r in toks)
    assert runner.batches == [[16, 2, 5], [1, 20], [23, 15, 1], [12, 64]]
    assert eng.alloc.num_free == 12 and eng.slots.num_free == 3 and not eng.seqs
    with pytest.raises(ValueError):
        eng.forced_step([("z", [99], [0])])                      # outside the vocabulary


@pytest.mark.parametrize("rows", [1, 16, 64])
def test_query_tiles_cover_every_row_once_in_order(rows):
    from mi355_decode import ops
    for lens in ([], [0], [1], [rows], [rows + 1, 0, 0, 2 * rows - 1], [0, 70, 3, 0, 129, rows, 0]):
        cu, want = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64), []
        for s, n in enumerate(lens):
            want += [[s, int(cu[s]) + a, min(rows, n - a)] for a in range(0, n, rows)]
        got = ops.query_tiles(cu, rows)
        assert got.dtype == np.int32 and got.flags.c_contiguous and got.shape == (len(want), 3) and got.tolist() == want


def test_step_fields_come_with_the_first_that_is_read():
    """Token ids, sizes and plans are there at once; the first other field brings all of them, once; an unknown one is an error."""
    from mi355_decode import hybrid_runner as HR
    calls = []

    def rest():
        calls.append(1)
        return {"positions": 1, "slot_mapping": 2, "block_tables": 3, "cu_seqlens": 4, "context_lens": None, "tok_seq": 5, "state_slots": 6,
                "tiles": 7}

    b = HR.StepBatch.behind(rest, torch.zeros(9, dtype=torch.int64), 3, True, None, 5, None, None, 8)
    assert (b.num_tokens, b.num_seqs, b.long_chunks, b.max_q_len, b.max_context, b.routes, b.keep_tail, b.tail) == \
        (9, 3, True, 5, 8, {}, False, None) and b.latent_plan is None and not calls
    assert b.context_lens is None and b.tiles == 7 and b.positions == 1 and b.tok_seq == 5 and calls == [1]
    with pytest.raises(AttributeError):
        b.no_such_field
    plain = HR.StepBatch(torch.zeros(2), 1, 2, 3, torch.zeros(3), 4, 5)
    assert plain.num_seqs == 2 and plain.tiles is None
    with pytest.raises(AttributeError):
        plain.no_such_field


def test_upload_keeps_values_shapes_and_types():
    from mi355_decode import ops
    src = [np.arange(5, dtype=np.int64) - 2, np.zeros((0,), np.int32), np.arange(6, dtype=np.int32).reshape(2, 3)[:, ::2], np.zeros((3, 0), np.int64)]
    for a, t in zip(src, ops.upload("cpu", *src)):
        assert t.is_contiguous() and tuple(t.shape) == a.shape and t.numpy().dtype == a.dtype and (t.numpy() == a).all()


# what the two forms took, us (staged, by tiles), chunk lengths, keys ahead of every chunk, (heads, kv heads, key size, value size), window
_WINDOW_SHAPES = [
    (90, 252, [2048] * 4, 0, (16, 4, 128, 128), 1024), (9, 31, [33] * 32, 0, (16, 4, 128, 128), 1024),
    (14, 28, [256], 0, (16, 4, 128, 128), 1024), (156, 738, [4096], 0, (16, 16, 128, 128), 4096),
    (25, 40, [300, 20, 150], 300, (16, 4, 128, 128), 1024), (13, 34, [2048], 0, (8, 8, 64, 64), 128),
    (636, 256, [1] * 31 + [8000], 0, (16, 4, 128, 128), 1024), (1700, 861, [1] * 31 + [8000], 0, (16, 4, 128, 128), 4096),
    (134, 75, [1] * 31 + [1000], 1000, (16, 4, 128, 128), 1024), (47, 26, [1] * 31 + [300], 1000, (4, 4, 64, 128), 1024),
    (99, 82, [512], 3000, (16, 4, 128, 128), 4096), (99, 47, [512], 3000, (8, 1, 128, 128), 4096),
    (79, 46, [512], 3000, (8, 8, 64, 64), 4096), (38, 30, [128], 1900, (16, 4, 128, 128), 1024),
]


@pytest.mark.parametrize("staged_us,tiles_us,lens,behind,sizes,window", _WINDOW_SHAPES)
def test_window_attention_takes_the_form_that_was_faster(monkeypatch, staged_us, tiles_us, lens, behind, sizes, window):
    """The dispatch of a prompt step's window attention at shapes where the two forms are far apart."""
    from types import SimpleNamespace
    from mi355_decode import hybrid_runner as HR, ops
    heads, kv, dim, vdim = sizes
    called, T = [], sum(lens)
    monkeypatch.setattr(ops, "rope_partial_kv_write", lambda *a: None)
    monkeypatch.setattr(ops, "sigmoid_window_attn_prefill", lambda *a, **k: called.append("staged"))
    monkeypatch.setattr(ops, "sigmoid_window_attn", lambda *a, **k: called.append("tiles"))
    width = [heads * dim, kv * dim, kv * vdim, heads]
    seg = {n: (sum(width[:i]), width[i]) for i, n in enumerate(("lq", "lk", "lv", "lg"))}
    meta = lambda *s, dt=torch.int32: torch.empty(*s, dtype=dt, device="meta")      # noqa: E731
    runner = SimpleNamespace(k_cache=[None], v_cache=[None], rotary=lambda d, b: None, linear=lambda x, w: x, key_splits=lambda b, s: {})
    spec = SimpleNamespace(heads=heads, kv_heads=kv, dim=dim, vdim=vdim, window=window, scale=1.0, rot_dims=0, rot_base=1.0)
    batch = HR.StepBatch(meta(T), meta(T), meta(T), None, meta(len(lens) + 1), meta(T), meta(len(lens)), meta(1, 3), True,
                         context_lens=meta(len(lens)), max_q_len=max(lens), max_context=max(lens) + behind)
    HR.WindowAttention(spec, SimpleNamespace(seg=seg, attn_temp=None, attn_bias=None, attn_o_w=None), runner, 0)(
        meta(T, -(-sum(width) // 8) * 8, dt=torch.bfloat16), batch)
    assert called == ["staged" if staged_us < tiles_us else "tiles"]


@pytest.mark.parametrize("rows,heads,kv_heads,rank,parts_us,one_us", [
    (1, 16, 8, 0, 14.9, 11.6), (256, 16, 8, 0, 146.2, 135.4), (32, 8, 4, 128, 34.8, 23.0), (128, 8, 4, 128, 65.1, 52.8), (64, 16, 8, 128, 64.1, 53.4),
    (256, 16, 8, 128, 158.4, 168.1), (32, 32, 16, 64, 62.1, 61.2), (64, 32, 16, 64, 96.2, 105.7), (256, 32, 16, 128, 270.3, 313.2),
    (128, 24, 12, 128, 129.2, 133.3), (256, 16, 16, 128, 161.5, 141.3), (1, 8, 4, 192, 25.6, 20.1), (256, 8, 4, 192, 99.1, 103.2),
    (1, 16, 8, 256, 24.7, 27.8), (256, 4, 2, 256, 67.3, 69.7), (1, 32, 16, 512, 29.0, 43.9), (256, 32, 16, 512, 280.3, 649.6)])
def test_delta_mixer_in_one_launch_where_that_is_faster(rows, heads, kv_heads, rank, parts_us, one_us):
    from mi355_decode import ops
    assert ops.delta_decode_pays(rows, heads, kv_heads, rank) == (one_us < parts_us)


def test_delta_mixer_in_one_launch_only_on_whole_pieces():
    """A norm's weight that starts inside a 16-byte piece (a view into a caller's flat float32 buffer) keeps the parts, which
    read it number by number."""
    from types import SimpleNamespace
    from mi355_decode.hybrid_runner import DeltaMixer
    spec = SimpleNamespace(heads=2, kv_heads=1, dim=128, vdim=128, per_channel=False)
    seg = {"q": (0, 128), "k": (128, 128), "v": (256, 256), "b": (512, 2), "a": (514, 2), "g": (520, 256)}
    flat = torch.ones(160)
    b = SimpleNamespace(long_chunks=False, num_tokens=3, num_seqs=3, max_q_len=1)
    for off in (0, 1, 2, 4, 8):
        lw = SimpleNamespace(seg=seg, conv_w=torch.zeros(512, 4, dtype=torch.bfloat16), head_norm=flat[off: off + 128])
        assert DeltaMixer(spec, lw, None, 0).one_launch(torch.zeros(3, 776, dtype=torch.bfloat16), b) == (off % 4 == 0)


@pytest.mark.parametrize("N,K,M,two_us,one_us", [
    (512, 1024, 16, 6.4, 4.4), (512, 1024, 32, 6.7, 5.1), (512, 1024, 64, 6.7, 7.1), (512, 2048, 17, 6.7, 7.2), (512, 2048, 64, 7.7, 10.1),
    (1024, 2048, 17, 7.0, 7.3), (1024, 2048, 33, 7.8, 9.5), (512, 512, 64, 6.2, 5.4), (2048, 1024, 64, 7.6, 7.2), (2048, 2048, 16, 7.1, 6.4),
    (2048, 2048, 33, 8.9, 9.7), (3072, 2048, 64, 10.2, 10.6), (4096, 2048, 64, 11.2, 10.7), (6208, 2048, 33, 11.9, 11.0), (8192, 2048, 1, 10.2, 8.6),
    (8192, 2048, 64, 14.4, 12.6), (16384, 2048, 32, 16.9, 18.6), (4096, 4096, 32, 11.8, 12.8)])
def test_gelu_goes_into_the_product_where_that_is_faster(N, K, M, two_us, one_us):
    from mi355_decode import ops
    assert ops.gelu_in_product(N, K, M) == (one_us < two_us)
