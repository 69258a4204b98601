"""Host-side geometry planning of the tiled decode GEMM (no GPU needed): the planner's choice
and the candidate list the tuner times must only name geometries the library builds, with K
splits the consumers can take."""
import pytest

from mi355_decode import ops

SHAPES = [  # N, K, split_k: the projections of the benchmark models and of their tensor-parallel slices
    (6144, 4096, True), (4096, 4096, True), (28672, 4096, False), (4096, 14336, True), (128256, 4096, False),
    (4608, 3584, True), (3584, 3584, True), (37888, 3584, False), (3584, 18944, True), (152064, 3584, False),
    (1280, 8192, True), (8192, 1024, True), (7168, 8192, False), (16032, 4096, False), (1536, 4096, True),
]
KW = {302, 304, 308, 402, 404}        # K split across the waves of a workgroup: up to 32 rows
BUILT = {16: {4, 8, 104, 108} | KW, 32: {4, 8, 104, 108} | KW,
         64: {8, 104, 108, 208, 210, 212, 214, 216, 302, 304, 402}, 128: {8, 210, 212, 214, 216, 302},
         256: {8, 210, 212, 214, 216, 302}}       # two row blocks of the 128-row geometries
# beyond 64 / 32 rows also row blocks of 64 (+ 1000: the 64-row geometries) / of 32 rows (+ 2000: the 32-row ones
# that exist for epilogues 0-2 on plain x)
ROW_BLOCKS = {1000 + t for t in BUILT[64]} | {2000 + t for t in (8, 104, 108, 302, 304, 402)}


@pytest.mark.parametrize("M", [1, 16, 17, 32, 33, 64, 65, 128, 129, 192, 256])
@pytest.mark.parametrize("N,K,split", SHAPES)
def test_candidates_are_built_geometries(M, N, K, split):
    cls = 16 if M <= 16 else 32 if M <= 32 else 64 if M <= 64 else 128 if M <= 128 else 256
    plan = ops.plan_linear_tiled(N, K, split, M)
    cands = ops.linear_tiled_candidates(N, K, split, M)
    if plan is None:
        assert cands == []
        return
    assert cands[0] == plan and len(set(cands)) == len(cands)
    for tiles, groups in cands:
        assert tiles in BUILT[cls] or (tiles in ROW_BLOCKS and M > ops.row_block_rows(tiles))
        ksl = ops.tiled_slice_width(M, tiles)
        assert ksl == ops.tiled_slice_width(min(M, ops.row_block_rows(tiles)), tiles % 1000)
        assert K % ksl == 0 and 1 <= groups <= min(K // ksl, 8)
        assert split or groups == 1
        assert ops.tiles_per_workgroup(tiles) in ((1, 2, 4) if tiles % 1000 in KW else (4, 8, 10, 12, 14, 16))
    if M <= 32:
        assert all(t < 1000 for t, _ in cands)


def test_narrow_slices_get_the_k_split_across_waves():
    """The qkv / o / gate_up slices of a Llama-3-70B rank on 8 GPUs at 16 rows: the forms with several
    waves per tile are among the candidates; a SwiGLU matrix never gets 8 waves per tile (its gate and
    up tiles must share a workgroup); wide matrices and more than 32 rows get none."""
    assert {t for t, _ in ops.linear_tiled_candidates(1280, 8192, True, 16)} >= {304, 308}
    assert (308, 1) in ops.linear_tiled_candidates(8192, 1024, False, 16)
    gu = {t for t, _ in ops.linear_tiled_candidates(7168, 8192, False, 16, swiglu=True)}
    assert gu & KW and 308 not in gu
    assert not {t for t, _ in ops.linear_tiled_candidates(28672, 4096, False, 32, swiglu=True)} & KW
    assert {t for t, _ in ops.linear_tiled_candidates(4096, 7168, False, 64)} & KW == {302, 304, 402}
    assert {t for t, _ in ops.linear_tiled_candidates(7168, 4096, False, 128, swiglu=True)} & KW == {302}
    # ... and in row blocks of 64 / 32 the forms of those row classes (a TP4 rank at 128 rows)
    rb = {t for t, _ in ops.linear_tiled_candidates(7168, 4096, False, 128, swiglu=True) if t >= 1000}
    assert {1302, 1304, 2302, 2304, 1008, 2008} <= rb and 2308 not in rb
    assert ops.row_block_rows(8) == 128 and ops.row_block_rows(1302) == 64 and ops.row_block_rows(2104) == 32
    assert ops.tiled_slice_width(128, 1302) == 512 and ops.tiled_slice_width(256, 2104) == 512
    assert ops.tiles_per_workgroup(1302) == 4 and ops.tiles_per_workgroup(2008) == 8
    assert ops.tiled_slice_width(16, 308) == 1024 and ops.tiled_slice_width(32, 404) == 512
    assert ops.tiled_slice_width(64, 304) == 512 and ops.tiled_slice_width(128, 302) == 256
    assert ops.tiles_per_workgroup(302) == 4 and ops.tiles_per_workgroup(308) == 1


def test_rows_beyond_the_kernels_have_no_plan():
    assert ops.plan_linear_tiled(4096, 4096, True, 257) is None
    assert ops.linear_tiled_candidates(4096, 4096, True, 257) == []
    assert ops.plan_linear_tiled(4096, 448, True, 32) is None          # K not a multiple of any slice width


def test_slice_widths_and_workgroup_tiles():
    assert [ops.tiled_slice_width(m, 8) for m in (16, 32, 64, 128)] == [1024, 1024, 512, 256]
    assert [ops.tiled_slice_width(m, 104) for m in (16, 32, 64, 128)] == [512, 512, 256, 128]
    assert ops.tiled_slice_width(64, 208) == 256 and ops.tiled_slice_width(64, 216) == 512
    assert ops.tiled_slice_width(128, 216) == 256
    assert [ops.tiles_per_workgroup(t) for t in (4, 8, 104, 108, 208, 210, 216)] == [4, 8, 4, 8, 8, 10, 16]
    assert ops.tiled_slice_width(64, 210) == 512 and ops.tiled_slice_width(128, 214) == 256
    # 2368 tiles (gate_up of Qwen2-7B): 16 per workgroup fill 148 CUs, 10 per workgroup 237
    assert (210, 1) in ops.linear_tiled_candidates(37888, 3584, False, 64, swiglu=True)


def test_row_blocks_count_as_workgroups():
    """129 .. 256 rows run as two row blocks: the same column blocks fill the chip with half the K split."""
    t128, g128 = ops.plan_linear_tiled(4096, 3584, True, 128)
    t256, g256 = ops.plan_linear_tiled(4096, 3584, True, 256)
    assert t128 == t256 == 8 and g256 < g128
    assert ops.tiled_slice_width(256, 8) == ops.tiled_slice_width(128, 8) == 256
    # a tensor-parallel rank's gate_up slice at 128 rows may split K (a SwiGLU-from-slabs kernel follows)
    assert any(g > 1 for _, g in ops.linear_tiled_candidates(7168, 4096, True, 128, swiglu=True))


def test_act_in_product_takes_what_the_tiles_take():
    import torch
    rows = lambda m, k, pad=0, dt=torch.bfloat16: torch.empty(m, k + pad, dtype=dt)[:, :k]      # noqa: E731
    w = torch.empty(8192, 2048, dtype=torch.bfloat16)
    yes = lambda x, w=w, act=ops.LINEAR_GELU_MUL: ops.act_in_product(x, w, act)                     # noqa: E731
    assert yes(rows(8192, 2048)) and yes(rows(8192, 2048, 8)) and yes(rows(2048, 2048))
    assert not yes(rows(8192, 2048, 4)) and not yes(rows(8192, 2048, 0, torch.float32)) and not yes(rows(8192, 2048, 0, torch.float16))
    assert not yes(torch.empty(8192, 2049, dtype=torch.bfloat16)[:, 1:]) and not yes(torch.empty(2048, 8192, dtype=torch.bfloat16).t())
    assert not yes(rows(8192, 2048), torch.empty(2048, 8192, dtype=torch.bfloat16).t())
    assert not yes(rows(8192, 2048), torch.empty(8200, 2048, dtype=torch.bfloat16)) and not yes(rows(8192, 1000), torch.empty(8192, 1000, dtype=torch.bfloat16))
    assert not yes(rows(128, 2048)) and not yes(rows(300, 2048))           # decoded rows; tiles that are mostly empty
    assert yes(rows(1500, 2048), act=ops.LINEAR_RELU2) and not yes(rows(1500, 2048))
    assert not yes(rows(640, 2048), act=ops.LINEAR_RELU2) and not yes(rows(1280, 2048), act=ops.LINEAR_RELU2)     # (1280: 46.6 us, two launches 45.6)
    # inputs at which the launch that is saved is a smaller part: sizes on both sides of the lines that were measured
    sizes = lambda m, n, k, act: ops._wide_pays(m, n, k, act)                                       # noqa: E731
    assert sizes(4096, 28672, 4096, ops.LINEAR_SILU_MUL) and sizes(512, 28672, 4096, ops.LINEAR_SILU_MUL) and not sizes(1280, 28672, 4096, ops.LINEAR_SILU_MUL)
    assert not sizes(1500, 16384, 4096, ops.LINEAR_GELU_MUL) and sizes(8192, 16384, 4096, ops.LINEAR_GELU_MUL)
    assert sizes(1789, 37888, 3584, ops.LINEAR_SILU_MUL) and not sizes(760, 32768, 4096, ops.LINEAR_SILU_MUL) and not sizes(2250, 16384, 3072, ops.LINEAR_SILU_MUL)
    assert not sizes(4096, 14336, 8192, ops.LINEAR_SILU_MUL) and not sizes(7168, 14336, 8192, ops.LINEAR_SILU_MUL)


def test_rows_past_rounds():
    f = ops.rows_past_rounds
    assert f(8193, 2048) == 8192 and f(8320, 6144) == 8192 and f(4224, 4096) == 4096 and f(2049, 8192) == 2048
    assert f(8192, 2048) == 0 and f(8321, 2048) == 0                       # none, more than the stream takes at its best
    assert f(4160, 3072) == 0 and f(2100, 4096) == 0 and f(8211, 3648) == 0   # tiles that leave a round part empty
    assert f(100, 65536) == 0 and f(1, 8192) == 0
    # few rows of wide outputs, where the stream of all the weights costs more: both sides of the line
    assert f(1088, 16384) == 0 and f(300, 65536) == 0 and f(2176, 57344) == 0 and f(2112, 57344) == 2048 and f(3200, 16384) == 3072 and f(2176, 8192) == 2048


def test_wide_product_rule():
    import torch
    x, w = torch.empty(8192, 2048, dtype=torch.bfloat16), torch.empty(6208, 2048, dtype=torch.bfloat16)
    out = torch.empty(8192, 6216, dtype=torch.bfloat16)
    f = ops.wide_product
    assert f(x, w) and f(x, w, out[:, :6208]) and f(x, torch.empty(5208, 2048, dtype=torch.bfloat16))
    assert not f(x, w, torch.empty(8192, 6209, dtype=torch.bfloat16)[:, :6208]) and not f(x, w, out[:, 4: 6212])
    assert not f(x, torch.empty(6144, 2048, dtype=torch.bfloat16)) and not f(x, torch.empty(6204, 2048, dtype=torch.bfloat16))
    assert not f(x[:1000], w[:2112]) and not f(x.float(), w.float()) and not f(x[:, :2040], w[:, :2040])


def test_heads_that_stream():
    """Sizes on both sides of the line that were measured, and no rows at all."""
    f = ops.head_streams
    assert f(1, 128256, 4096) and f(64, 128256, 4096) and f(64, 152064, 3584) and f(64, 64128, 4096) and f(32, 16032, 8192) and f(32, 50272, 1024)
    assert not f(0, 128256, 4096) and not f(65, 128256, 4096) and not f(33, 16032, 8192) and not f(64, 38016, 3584) and not f(33, 50272, 1024)


@pytest.mark.parametrize("M,N,K,takes", [(6189, 3648, 2048, False), (7168, 5184, 2048, False), (8211, 3648, 2048, True), (8192, 6176, 2048, True),
                                         (4096, 5208, 2048, False), (6189, 10352, 4096, False), (8192, 4544, 3584, False), (6000, 2112, 1024, True)])
def test_wide_products_where_they_were_the_faster_way(M, N, K, takes):
    """Sizes on both sides of the line that were measured."""
    assert (ops.product_route(M, N, K) == -1) == takes


def test_product_route_says_what_the_rules_say_and_is_worked_out_once():
    import torch
    seen = set()
    for M in (257, 1000, 4100, 8192, 8211):
        x = torch.empty(M, 2048, dtype=torch.bfloat16)
        for N in (2048, 3648, 6176, 6204, 8192):
            want = -1 if ops.wide_product(x, torch.empty(N, 2048, dtype=torch.bfloat16)) else ops.rows_past_rounds(M, N)
            assert ops.product_route(M, N, 2048) == want
            seen.add(min(want, 1))
    assert seen == {-1, 0, 1}
    misses = ops.product_route.cache_info().misses
    assert ops.product_route(8192, 6176, 2048) == -1 and ops.product_route.cache_info().misses == misses


def test_gated_activation_codes_are_the_abis():
    """What the mixtures' and the row kernels' entries read; linear_act counts its activations by names of its own."""
    assert ops._gate_act(None) == (0, 0.0) and ops._gate_act(7.0) == (1, 7.0)
    assert (ops.ACT_SILU, ops.ACT_SIGMOID) == (0, 1)
    assert (ops.LINEAR_RELU2, ops.LINEAR_GELU_MUL, ops.LINEAR_SILU_MUL, ops.LINEAR_LIMITED_MUL, ops.LINEAR_NONE) == (0, 1, 2, 3, 4)


@pytest.mark.parametrize("in_product", [True, False])
def test_prompt_layers_hold_gate_and_up_rows_only_where_no_product_takes_the_unit(monkeypatch, in_product):
    """[tokens, 2 ff] is the largest buffer of a prompt step: made once, and only by the two-launch way."""
    import torch
    from types import SimpleNamespace
    from mi355_decode.model_runner import ModelRunner
    r, made, real = object.__new__(ModelRunner), [], torch.empty
    r.w = SimpleNamespace(layers=[SimpleNamespace(input_norm=None, post_norm=None, qkv_b=None)] * 3)
    r.eps, r.F, r.dtype, r.device, r.mlp_sharded = 1e-6, 24, torch.float32, "cpu", False
    r._product = r._allreduce = lambda *a: None
    r._rm = lambda i, kind: torch.ones(48, 16)
    for name in ("rms_norm", "fused_add_rms_norm", "linear_act"):
        monkeypatch.setattr(ops, name, lambda *a, **k: None)
    monkeypatch.setattr(ops, "act_in_product", lambda *a: in_product)
    monkeypatch.setattr(ops, "silu_and_mul", lambda gu, out: out.copy_(gu[:, :24]))
    monkeypatch.setattr(torch, "empty", lambda *a, **k: made.append(a) or real(*a, **k))
    x, act = torch.ones(5, 16), torch.zeros(5, 24)
    r._layers(5, None, x, None, None, None, act, None, lambda *a: None)
    assert made == ([] if in_product else [(5, 48)]) and (act == (0 if in_product else 16)).all()
