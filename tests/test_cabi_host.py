"""CPU-side checks of the C-ABI library and the host logic above it (no kernel is launched).

* libladder_hip.so loads and exports every symbol include/ladder_hip.h declares, and the ctypes
  prototypes of gpt_fast/_hip.py cover exactly that set;
* argument validation answers before anything touches the device;
* the configuration registry reproduces the reference's shapes (gpt_ladder_TP.py:20-207) and the
  per-rank sizes of the benchmark configurations;
* modules built on the meta device carry the reference's parameter names and shapes;
* bytes-per-step accounting used for the roofline."""
import ctypes
import os
import re

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols():
    text = open(os.path.join(ROOT, "include", "ladder_hip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(lr_[a-z0-9_]+)\s*\(", text)))


@pytest.fixture(scope="module")
def lib():
    from gpt_fast import _hip

    if not os.path.exists(_hip.lib_path()):
        pytest.fail(f"{_hip.lib_path()} has not been built (python ladder-residual-inference_amd/build.py)")
    return _hip.load()


def test_library_exports_every_declared_symbol(lib):
    from gpt_fast import _hip

    names = declared_symbols()
    assert len(names) >= 20
    raw = ctypes.CDLL(_hip.lib_path())
    missing = [n for n in names if not hasattr(raw, n)]
    assert not missing, missing
    assert sorted(_hip.exported_names()) == names


def test_version_and_error_strings(lib):
    assert lib.lr_version() >= 1
    seen = set()
    for code in range(0, -7, -1):
        s = lib.lr_error_string(code)
        assert s and s.decode()
        seen.add(s)
    assert len(seen) >= 6, "every error code has its own message"


def test_validation_precedes_any_device_work(lib):
    # null / misaligned pointers and impossible shapes are refused on the host (no GPU here)
    E_NULL, E_ALIGN, E_SHAPE = -1, -2, -3
    assert lib.lr_add(None, None, 1.0, None, 16, None) == E_NULL
    assert lib.lr_add(8, 16, 1.0, 32, 16, None) == E_ALIGN
    assert lib.lr_linear(None, 0, None, None, 0, 1, 8, 8, 0, None) == E_NULL
    assert lib.lr_linear(64, 8, 128, 256, 8, 0, 8, 8, 0, None) == E_SHAPE
    assert lib.lr_argmax(None, 0, None, 1, 8, None) == E_NULL
    from gpt_fast._hip import _Projection, EPI_SWIGLU
    import ctypes
    one = (_Projection * 1)(_Projection(64, 8, 128, 256, 8, 8, 8, 0))
    ptr = ctypes.cast(one, ctypes.c_void_p)
    assert lib.lr_linear_multi(None, 1, 1, None) == E_NULL
    assert lib.lr_linear_multi(ptr, 3, 1, None) == E_SHAPE          # at most two projections
    assert lib.lr_linear_multi(ptr, 1, 65, None) == -4              # more than 64 rows: unsupported
    one[0].epilogue = EPI_SWIGLU
    one[0].N = 7                                                    # [up; gate] rows come in pairs
    assert lib.lr_linear_multi(ptr, 1, 1, None) == E_SHAPE
    one[0].N, one[0].K = 8, 12                                      # K % 8
    assert lib.lr_linear_multi(ptr, 1, 1, None) == E_SHAPE          # ldx < K
    one[0].ldx = 16
    assert lib.lr_linear_multi(ptr, 1, 1, None) == E_ALIGN
    # attention beside a projection: attention arguments as lr_attn_decode, then what it has no kernel for
    one[0] = _Projection(64, 8, 128, 256, 8, 8, 8, 0)

    def beside(q, proj, M, epi=0, scratch_bytes=1 << 30):
        one[0].epilogue = epi
        return lib.lr_attn_decode_beside(q, 1024, 128, 256, 512, 1024, 1024, 4, 8, 1, 128, 64, 2048, scratch_bytes,
                                         proj, M, None)

    assert beside(None, ptr, 4) == E_NULL
    assert beside(64, None, 4) == E_NULL
    assert beside(64, ptr, 0) == E_SHAPE
    assert beside(64, ptr, 17) == -4                                # the 16-row band only
    assert beside(64, ptr, 4, epi=2) == -4                          # a projection that writes the cache
    assert beside(64, ptr, 4, scratch_bytes=16) == E_SHAPE
    # the prefill's q/k/v projection with the rotation and the cache writes in its output pass
    from gpt_fast._hip import _RopeKv
    rope = _RopeKv(64, 128, 192, 256, None, 8, 1, 128, 64, 64)          # N = (8 + 2) * 128 = 1280

    def fused(x=64, ldx=64, ldy=1280, M=8, K=64, S=4, r=rope):
        return lib.lr_linear_rope_kv(x, ldx, 128, 256, ldy, M, K, S, None if r is None else ctypes.byref(r), None)

    assert fused(x=None) == E_NULL
    assert fused(r=None) == E_NULL
    assert fused(M=9) == E_SHAPE                                        # whole sequences of S tokens
    assert fused(ldy=1272) == E_SHAPE                                   # ldy < N
    assert fused(ldy=1284) == E_ALIGN
    assert fused(K=60, ldx=64) == E_ALIGN
    assert fused(r=_RopeKv(64, None, 192, 256, None, 8, 1, 128, 64, 64)) == E_NULL      # no positions
    assert fused(r=_RopeKv(64, 128, 192, 256, None, 8, 1, 124, 64, 64), ldy=1240) == E_ALIGN   # head_dim % 8
    from gpt_fast._hip import _ProjectionFp8
    one8 = (_ProjectionFp8 * 1)(_ProjectionFp8(64, 16, 128, 192, 256, 8, 8, 16, 0))
    ptr8 = ctypes.cast(one8, ctypes.c_void_p)
    assert lib.lr_linear_fp8_multi(None, 1, 1, None) == E_NULL
    assert lib.lr_linear_fp8_multi(ptr8, 1, 17, None) == -4           # up to 16 rows
    assert lib.lr_linear_fp8_multi(ptr8, 3, 1, None) == E_SHAPE
    one8[0].K = 24                                                    # 16 weights per lane and load
    assert lib.lr_linear_fp8_multi(ptr8, 1, 1, None) == E_SHAPE       # ldx < K
    one8[0].ldx = 24
    assert lib.lr_linear_fp8_multi(ptr8, 1, 1, None) == E_ALIGN
    one8[0].K, one8[0].ldx, one8[0].scales = 16, 16, None
    assert lib.lr_linear_fp8_multi(ptr8, 1, 1, None) == E_NULL
    assert lib.lr_ladder_decode_step(None, 1, None, None, None, 0, None, 0, None, None, 0, 0, 0, None, 0, None) == E_NULL
    assert lib.lr_ladder_decode_step_fp8(None, 1, None, None, None, 0, None, 0, None, None, 0, 0, 0, None, 0, None) == E_NULL
    assert lib.lr_ladder_step_workspace_bytes(None, 1) == 0


def test_missing_library_is_an_error(monkeypatch):
    from gpt_fast import _hip

    monkeypatch.setattr(_hip, "_lib", None)
    monkeypatch.setattr(_hip, "_LIB_PATH", os.path.join(ROOT, "no_such_dir", "libladder_hip.so"))
    with pytest.raises(_hip.LadderHipError):
        _hip.load()


def test_registry_matches_reference_shapes():
    from gpt_fast.config import ModelArgs, args_from_name

    a = args_from_name("ladder", "llama-3-8b")
    assert (a.dim, a.n_layer, a.n_head, a.n_local_heads, a.intermediate_size, a.vocab_size) == \
        (4096, 32, 32, 8, 14336, 128256)
    assert a.head_dim == 128 and a.rope_base == 500000
    # default intermediate size: round_up(int(8 * dim / 3), 256)   (gpt_ladder_TP.py:56-60)
    b = ModelArgs(dim=1000, n_head=8, n_layer=1)
    assert b.intermediate_size == 2816 and b.n_local_heads == 8 and b.head_dim == 125
    # one tensor-parallel rank of Ladder-70B at TP = 8
    c = args_from_name("ladder", "ladder-70b-tp8")
    assert (c.tp_world_size, c.n_head_local, c.n_kv_local, c.ffn_local, c.output_rows) == (8, 8, 1, 3584, 16032)
    d = args_from_name("ladder", "ladder-405b-tp8")
    assert (d.dim, d.n_layer, d.n_head_local, d.n_kv_local, d.ffn_local) == (16384, 126, 16, 1, 6656)
    with pytest.raises(AssertionError):
        ModelArgs(dim=512, n_head=8, n_layer=1, intermediate_size=1022, tp_world_size=4)   # not divisible by tp
    from gpt_fast.utils import Attention

    with pytest.raises(AssertionError), torch.device("meta"):   # heads not divisible by tp (utils.py:155-162)
        Attention(ModelArgs(dim=512, n_head=8, n_local_heads=2, n_layer=1, intermediate_size=1024, tp_world_size=4))


@pytest.mark.parametrize("family", ["ladder", "dense", "desync", "parallel"])
def test_meta_modules_have_reference_parameter_names(family):
    import benchmark as bm
    from gpt_fast.config import ModelArgs
    from oracle import ladder_oracle as O

    kw = dict(block_size=64, vocab_size=512, n_layer=2, n_head=4, n_local_heads=2, dim=256, intermediate_size=512)
    cls = {"ladder": bm.GPTLadder, "dense": bm.GPTDense, "desync": bm.GPTDesync, "parallel": bm.GPTParallel}[family]
    with torch.device("meta"):
        model = cls(ModelArgs(**kw))
    got = {n: tuple(p.shape) for n, p in model.named_parameters()}
    want = dict(O.param_shapes(O.OracleConfig(**kw), family))
    assert got == want


def test_virtual_tp_builds_one_rank_without_a_process_group(monkeypatch):
    from gpt_fast import maybe_init_dist, tp

    assert maybe_init_dist() == 0
    tp.set_virtual_tp(8, 3)
    try:
        assert tp.get_tp_world_size() == 8 and tp.get_tp_rank() == 3
    finally:
        tp.set_virtual_tp(1, 0)
    with pytest.raises(AssertionError):
        tp.set_virtual_tp(4, 4)
    assert not torch.distributed.is_initialized()
    monkeypatch.setenv("WORLD_SIZE", "2")     # a multi-process launch is refused, never silently run
    with pytest.raises(RuntimeError):
        maybe_init_dist()


def test_shard_vocab_flag_reaches_the_model_shape():
    """benchmark.py --virtual_tp N --shard_vocab: the lm_head of the unsharded registry names is built at
    vocab_size / N rows (the reference's flag surface is benchmark.py:498-518; it replicates the head)."""
    import benchmark as bm
    from gpt_fast import tp
    from gpt_fast.config import args_from_name

    args = bm.build_parser().parse_args(["--model_name", "gpt_ladder:70B", "--prompt_length", "8", "--virtual_tp", "8",
                                         "--shard_vocab"])
    assert args.shard_vocab and args.virtual_tp == 8
    tp.set_virtual_tp(args.virtual_tp, args.tp_rank, args.shard_vocab)
    try:
        c = args_from_name("ladder", "70B")
        assert c.tp_world_size == 8 and c.shard_vocab and c.output_rows == c.vocab_size // 8
        assert c.n_head_local == 8 and c.n_kv_local == 1 and c.ffn_local == 3584
    finally:
        tp.set_virtual_tp(1, 0)
    c = args_from_name("ladder", "70B")
    assert not c.shard_vocab and c.output_rows == c.vocab_size
    assert not bm.build_parser().parse_args(["--model_name", "gpt_ladder:70B", "--prompt_length", "8"]).shard_vocab


def test_bytes_per_step_accounting():
    import benchmark as bm
    from gpt_fast.config import args_from_name

    c = args_from_name("ladder", "ladder-70b-tp8")
    b0 = bm.decode_bytes_per_step(c, 1, 2048)
    # weights 17.378 GB + valid KV + KV write + embedding row + logits: 17.462 GB at position 2048
    assert abs(b0 - 17.462e9) < 0.003e9
    # one more position costs one more K and V row per layer
    assert bm.decode_bytes_per_step(c, 1, 2049) - b0 == 80 * 2 * 128 * 2
    # a second sequence adds its KV, embedding row and logits, not the weights
    assert bm.decode_bytes_per_step(c, 2, 2048) - b0 < 0.1e9


def _desc(**over):
    from gpt_fast import _hip

    kw = dict(dim=256, n_layer=2, n_head=4, n_kv_head=2, head_dim=64, ffn=512, out_rows=512, vocab=512, smax=64,
              block_size=64, eps=1e-5, attention_workgroups=0, tok_embeddings=4096, norm=4096, output=4096,
              freqs_cis=4096, layers_dev=4096)
    kw.update(over)
    return _hip.LadderModelDesc(**kw)


def test_step_descriptor_is_validated_on_the_host(lib):
    """Shapes the one-kernel step must refuse are refused before any device is looked at (no GPU here)."""
    import ctypes

    E_NULL, E_SHAPE, E_UNSUPPORTED = -1, -3, -4
    # (the workspace pointer is misaligned on purpose: where a GPU is present a descriptor that passes validation is
    # then refused with LR_E_ALIGN instead of being initialised at a made-up address)
    init = lambda d, b=1: lib.lr_ladder_step_init(ctypes.byref(d), b, 8, 1 << 20, None)
    # a cache longer than the RoPE table: positions beyond block_size would read past the end of freqs_cis
    assert init(_desc(smax=72, block_size=64)) == E_SHAPE
    assert lib.lr_ladder_step_workspace_bytes(ctypes.byref(_desc(smax=72, block_size=64)), 1) == 0
    assert init(_desc(smax=64, block_size=60)) != E_SHAPE          # the cache length is rounded up to 8
    assert init(_desc(n_head=5)) == E_SHAPE                        # q heads not a multiple of kv heads
    assert init(_desc(), b=3) == E_UNSUPPORTED                     # batch: 1 or 2
    assert init(_desc(head_dim=48)) == E_UNSUPPORTED
    assert init(_desc(dim=20000)) == E_UNSUPPORTED


def test_load_hook_fuses_separate_projections():
    """utils.py:178-185: checkpoints with wq / wk / wv load into the fused wqkv, rows [q; k; v]."""
    from gpt_fast.config import ModelArgs
    from gpt_fast.utils import Attention

    cfg = ModelArgs(dim=64, n_head=4, n_local_heads=2, n_layer=1, intermediate_size=128)
    att = Attention(cfg)
    g = torch.Generator().manual_seed(0)
    wq, wk, wv = (torch.randn(r, 64, generator=g) for r in (64, 32, 32))
    wo = torch.randn(64, 64, generator=g)
    att.load_state_dict({"wq.weight": wq, "wk.weight": wk, "wv.weight": wv, "wo.weight": wo})
    assert torch.equal(att.wqkv.weight, torch.cat([wq, wk, wv])) and torch.equal(att.wo.weight, wo)
    # an already fused checkpoint passes through untouched
    att2 = Attention(cfg)
    att2.load_state_dict(att.state_dict())
    assert torch.equal(att2.wqkv.weight, att.wqkv.weight)


def test_setup_caches_refuses_a_sequence_longer_than_block_size():
    import benchmark as bm
    from gpt_fast.config import ModelArgs

    with torch.device("meta"):
        model = bm.GPTLadder(ModelArgs(block_size=64, vocab_size=512, n_layer=1, n_head=4, dim=256))
    with pytest.raises(ValueError):
        model.setup_caches(1, 65)


FAMILIES = [("ladder", "ladder-70b-tp8"), ("dense", "ladder-8b"), ("desync", "ladder-8b"), ("parallel", "ladder-8b"),
            ("lasivik", "lasivik-8b"), ("gepolix", "gepolix-8b")]


def meta_model(family, name):
    import gpt_fast

    with torch.device("meta"):
        m = getattr(gpt_fast, "GPT" + family.capitalize()).from_name(name).to(torch.bfloat16)
    m.max_batch_size, m.max_seq_length = 96, 1024
    if family in ("lasivik", "gepolix"):
        m._build_caches(96, 1024, torch.bfloat16, torch.device("meta"))
    return m


@pytest.mark.parametrize("family,name", FAMILIES)
@pytest.mark.parametrize("B,S", [(1, 1), (32, 1), (1, 20), (2, 16), (33, 1), (64, 1), (96, 1), (1, 33), (1, 777), (4, 512)])
def test_memory_for_partial_sums_is_what_the_products_of_a_step_can_use(lib, family, name, B, S):
    """Enough for every product to be divided as with all the memory it could ask for, and no more than that."""
    from gpt_fast import _hip

    model = meta_model(family, name)
    for model.last_logits_only in (False, True):
        products = set(model._products(B, S))
        assert len(products) >= 4
        ws = model._new_workspace(B, S)
        if B * S <= 32:
            assert ws.sums is None and not any(lib.lr_linear_scratch_bytes(p[0]) for p in products if p[0] == B * S)
            continue
        held = ws.sums.numel()
        plans = [(p, _hip.linear_plan(*p)) for p in products if lib.lr_linear_scratch_bytes(p[0])]
        assert held == max(256, *(q.sums_bytes for _, q in plans)) <= lib.lr_linear_scratch_bytes(B * S)
        for p, full in plans:
            assert bytes(full) == bytes(_hip.linear_plan(*p, scratch_bytes=held))
        if S == 1 and B <= 64:
            assert held <= 16 << 20


# Products of models' weights in us, by tile (rows, columns) and pieces of K, measured one after the other with weights from HBM: the
# choice that costs fitted to fewer of them made, and the ones near the best (where tiles of 160, 192 and 224 rows are among these, all
# of the product's measured again together).
MEASURED_PRODUCTS = [
    # M, N, K, pair, MiB for pieces
    (1700, 1024, 16, False, 64, {(128, 128, 1): 5.1, (64, 128, 1): 4.2}),
    (900, 2048, 16, False, 0, {(128, 128, 1): 5.1, (64, 128, 1): 4.2}),
    (200, 8192, 512, False, 64, {(128, 128, 1): 7.2, (64, 128, 1): 6.0}),
    (512, 4096, 512, False, 64, {(128, 128, 1): 7.3, (64, 128, 1): 6.3}),
    (129, 4096, 22528, False, 64, {(256, 256, 12): 64.2, (128, 256, 8): 57.0, (128, 128, 4): 55.9, (160, 128, 8): 53.0}),
    (1501, 7168, 8192, True, 64, {(256, 256, 1): 162.5, (128, 256, 3): 156.7, (192, 256, 1): 138.4}),
    (257, 2048, 12288, False, 64, {(128, 256, 10): 29.8, (128, 128, 5): 28.0, (160, 128, 8): 27.4, (192, 128, 8): 26.8}),
    (4100, 8192, 1024, False, 64, {(256, 256, 1): 84.8, (256, 256, 4): 81.0, (192, 256, 1): 70.0}),
    (1315, 2048, 5120, False, 64, {(128, 256, 2): 40.6, (128, 128, 1): 37.6, (192, 128, 2): 35.4}),
    (3002, 7168, 8192, True, 0, {(256, 256, 1): 332.5, (128, 256, 1): 289.6, (192, 256, 1): 275.1}),
    (2630, 6160, 2048, False, 0, {(128, 256, 1): 84.5, (128, 128, 1): 73.5, (192, 128, 1): 61.5}),
    (6004, 4096, 4096, True, 0, {(256, 256, 1): 178.3, (128, 256, 1): 165.1, (192, 256, 1): 155.3}),
    (9205, 2048, 8192, False, 0, {(128, 256, 1): 278.1, (128, 128, 1): 255.8, (192, 128, 1): 227.4}),
    (520, 28672, 4096, True, 0, {(128, 256, 1): 167.0, (128, 128, 1): 153.4, (160, 256, 1): 126.9}),
    # and what those costs had won over the ones before
    (128, 2048, 2048, False, 64, {(64, 128, 8): 12.4, (64, 128, 4): 10.4, (64, 128, 3): 10.1}),
    (900, 2048, 2048, False, 64, {(128, 128, 1): 15.3, (64, 128, 1): 12.8}),
    (128, 3072, 2048, False, 64, {(64, 128, 1): 17.2, (64, 128, 4): 13.3, (64, 128, 5): 13.0}),
    (128, 4096, 14336, False, 64, {(64, 128, 8): 38.3, (128, 128, 8): 32.8}),
    (128, 28672, 4096, True, 64, {(64, 128, 1): 65.8, (128, 128, 1): 54.8}),
    (136, 1280, 8192, False, 64, {(64, 128, 8): 15.5, (160, 128, 16): 16.5}),
    (145, 2048, 5120, False, 64, {(64, 128, 5): 16.2, (160, 128, 10): 17.9}),
    (160, 2048, 10240, False, 64, {(128, 128, 8): 19.8, (160, 128, 16): 20.8}),
    (9205, 2560, 2048, False, 64, {(256, 256, 2): 95.6, (128, 256, 1): 85.9, (192, 256, 1): 80.2}),
]


@pytest.mark.parametrize("M,N,K,pair,mib,times", MEASURED_PRODUCTS)
def test_the_plan_takes_no_tiles_that_measured_slower(lib, M, N, K, pair, mib, times):
    """Within 3 % of the fastest, the difference that two runs of one product may show."""
    from gpt_fast import _hip

    plan = _hip.linear_plan(M, N, K, pair, mib << 20)
    assert times[(plan.tile_rows, plan.tile_cols, plan.pieces)] <= 1.03 * min(times.values())


@pytest.mark.parametrize("M,N,K,pair,mib,times", [
    (112, 8192, 15360, False, 64, {(128, 128, 3): 66.9, (128, 128, 4): 55.8}),
    (112, 8192, 12288, False, 64, {(128, 128, 3): 54.1, (128, 128, 4): 48.3}),
    (112, 5120, 13824, False, 64, {(128, 128, 5): 40.0, (128, 128, 6): 36.2}),
    (112, 6144, 17920, False, 64, {(128, 128, 4): 58.9, (128, 256, 8): 52.7, (128, 128, 5): 51.3}),
    (112, 20480, 5120, True, 64, {(128, 128, 1): 61.3, (128, 256, 3): 52.6}),
    (112, 21504, 7168, True, 64, {(128, 128, 1): 79.4, (128, 256, 3): 72.3}),
    (112, 24576, 8192, False, 64, {(128, 128, 1): 86.0, (128, 256, 2): 114.0}),
    (112, 16384, 12288, False, 64, {(128, 128, 2): 92.5, (128, 256, 3): 112.4})])
def test_the_plan_takes_the_ring_of_three_where_it_measured_faster(lib, M, N, K, pair, mib, times):
    """Against the tiles beside it: it is the slower one where it leaves CUs without work."""
    test_the_plan_takes_no_tiles_that_measured_slower(lib, M, N, K, pair, mib, times)


# (rows of a prompt, of a decode step; us of a measured one and two products beside the rule)
@pytest.mark.parametrize("name,S,B,two", [
    ("ladder-8b", 64, 0, True), ("ladder-8b", 150, 0, True), ("ladder-8b", 0, 70, True), ("ladder-8b", 0, 160, True), ("ladder-8b", 190, 0, False),
    ("ladder-1b", 64, 0, True), ("ladder-1b", 150, 0, True), ("ladder-1b", 0, 70, False), ("ladder-1b", 0, 160, False),
    ("ladder-70b-tp8", 64, 0, True), ("ladder-70b-tp8", 0, 70, False), ("ladder-70b-tp8", 4100, 0, True),
    ("llama-3.2-3b", 30, 0, True), ("llama-3.2-3b", 100, 0, False), ("llama-3.2-3b", 150, 0, False), ("llama-3.2-3b", 0, 70, False),
    ("llama-3.2-3b", 0, 160, False), ("7B", 40, 0, True), ("7B", 150, 0, False), ("70B", 0, 160, True), ("ladder-405b-tp8", 64, 0, False),
    ("ladder-405b-tp8", 0, 100, False)])
def test_parallel_blocks_take_the_form_that_measured_faster(lib, name, S, B, two):
    """And hold memory for the two products' sums only where they run."""
    model = meta_model("parallel", name)
    B, S = (B, 1) if B else (1, S)
    assert model._in_parts(B, S) == two
    nqkv = (model.config.n_head_local + 2 * model.config.n_kv_local) * model.config.head_dim
    assert any(N == nqkv for rows, N, K, pair in model._products(B, S) if rows == B * S) == two


def test_the_plans_us_are_those_of_its_refusals(lib):
    from gpt_fast import _hip

    assert _hip.linear_plan_us(64, 4096, 4096) > 0 and _hip.linear_plan_us(64, 28672, 4096, True) > _hip.linear_plan_us(64, 4096, 4096)
    for bad in ((0, 64, 64), (64, 0, 64), (64, 64, 0), (64, 65, 64, True), (64, 64, 60)):
        assert _hip.linear_plan_us(*bad) == 0.0


def test_a_model_without_bf16_projections_holds_no_memory_for_partial_sums(lib):
    from gpt_fast.quantize import quantize_model_fp8

    model = meta_model("ladder", "ladder-70b-tp8")
    assert model._new_workspace(48, 1).sums is not None      # (also where the model is quantised after its first use)
    quantize_model_fp8(model)
    for B, S in ((48, 1), (1, 777)):
        assert model._new_workspace(B, S).sums is None


def test_only_prompts_whose_blocks_keep_both_outputs_pieces_hold_memory_for_both(lib):
    """lr_ladder_block's: all-ladder models on bf16 weights.  Others, with a bf16 head or whole, hold one piece of memory."""
    import gpt_fast
    from gpt_fast.quantize import quantize_model_fp8

    apart = lambda model: (lambda ws: ws.sums is not None and ws.sums is not ws.sums_mlp)(model._new_workspace(1, 777))
    assert apart(meta_model("ladder", "ladder-8b"))
    quantised = quantize_model_fp8(meta_model("ladder", "ladder-8b"), include_output=False)
    assert quantised._new_workspace(1, 777).sums is not None and not apart(quantised)
    assert not apart(meta_model("dense", "ladder-8b"))
    partial = meta_model("ladder", "ladder-8b")
    partial.config.ladder_layers = [0, 1]
    assert partial._new_workspace(1, 777).sums is not None and not apart(partial)


@pytest.mark.parametrize("family,name", FAMILIES[:3])
@pytest.mark.parametrize("B", [33, 64, 65, 96])
def test_partial_sums_of_the_mlp_are_limited_where_that_was_measured(lib, family, name, B):
    """Memory of its own beside the attention's: a part as large up to 64 rows, all that the products can use above."""
    ws = meta_model(family, name)._new_workspace(B, 1)
    assert ws.sums_mlp is not ws.sums and ws.sums_mlp._base is None
    assert ws.sums_mlp.numel() == (min(ws.sums.numel(), 200 << 15) if B <= 64 else ws.sums.numel())


@pytest.mark.parametrize("family", ["ladder", "parallel"])
@pytest.mark.parametrize("name", ["ladder-1b", "ladder-8b", "ladder-70b-tp8", "ladder-405b-tp8"])
@pytest.mark.parametrize("B", [16, 17, 32, 33, 64, 65])
def test_shared_grids_of_a_decode_step_hold_the_memory_that_their_products_can_use(lib, family, name, B):
    """The up/gate product beside the attention, and in a ladder block wo beside w2: divided as with all the memory they could ask for."""
    from gpt_fast import _hip

    model = meta_model(family, name)
    c, ws = model.config, model._new_workspace(B, 1)
    if B in (16, 65) or (family, B > 32) == ("parallel", True):
        assert ws.pair_sums == []
        return
    held = [t.numel() for t in ws.pair_sums]
    up = (B, 2 * c.ffn_local, c.dim, True)
    assert bytes(_hip.linear_plan(*up, scratch_bytes=held[0])) == bytes(_hip.linear_plan(*up, scratch_bytes=64 << 20))
    if family == "ladder":
        two = lib.lr_linear_pieces_two_bytes(B, c.dim, c.n_head_local * c.head_dim, c.ffn_local)
        assert len(held) == 2 and ws.pair_sums[0] is not ws.pair_sums[1] and 0 < two <= min(held)
    assert max(held) <= 16 << 20


def test_swiglu_projection_of_many_rows_refuses_what_its_two_calls_refuse(lib):
    """More than 64 rows on a small grid are specified as lr_linear into `scratch` and lr_swiglu: scratch of the projection's
    size, multiples of 8 columns, and no more rows than lr_swiglu takes -- with memory for partial sums or without."""
    E_NULL, E_ALIGN, E_SHAPE = -1, -2, -3
    p, big = 4096, 1 << 40

    def call(M, N, ldy, scratch, n, sums):
        return lib.lr_linear_swiglu_out_scratch(p, 64, p, p, ldy, M, N, 64, scratch, n, sums, 1 << 20 if sums else 0, None)

    for sums in (None, p):
        assert call(65, 48, 24, None, 0, sums) == E_NULL
        assert call(65, 48, 24, 8, big, sums) == E_ALIGN
        assert call(65, 48, 24, p, 2 * 65 * 48 - 1, sums) == E_SHAPE
        assert call(65, 36, 24, p, big, sums) == E_ALIGN            # 18 pairs
        assert call(65, 48, 25, p, big, sums) == E_ALIGN            # rows of 25 elements
        assert call(65535 * 64 + 1, 48, 24, p, big, sums) == E_SHAPE
    assert lib.lr_linear_swiglu_out(p, 64, p, p, 24, 65, 36, 64, p, big, None) == E_ALIGN


def test_bands_end_where_products_with_partial_sums_begin(lib):
    from gpt_fast import _hip

    assert lib.lr_linear_scratch_bytes(_hip.BANDS_TO) == 0 and lib.lr_linear_scratch_bytes(_hip.BANDS_TO + 1) > 0


def test_only_contiguous_device_memory_is_handed_on_for_partial_sums():
    from gpt_fast import _hip

    assert _hip._scratch_args(None) == (None, 0)
    for t in (torch.empty(64, dtype=torch.uint8), torch.empty(1, dtype=torch.uint8).expand(64), torch.empty(64)[::2]):
        with pytest.raises(AssertionError):
            _hip._scratch_args(t)


def test_gemm_plan_covers_every_tile_and_refuses_sizes_beyond_its_integers(lib):
    from gpt_fast import _hip

    p = _hip._LinearPlan()
    big = 0x7fffffff
    for M, N, K in ((big, 8, 8), (8, big, 8), (8, 8, big - 7), (big - 255, 8, 8), (1 << 30, 1 << 30, 8)):
        assert lib.lr_linear_plan(M, N, K, 0, 0, ctypes.byref(p)) == -4, (M, N, K)
    assert lib.lr_linear_plan(8, 7, 8, 1, 0, ctypes.byref(p)) == -3 and lib.lr_linear_plan(0, 8, 8, 0, 0, ctypes.byref(p)) == -3
    assert lib.lr_linear_plan(8, 8, 12, 0, 0, ctypes.byref(p)) == -2 and lib.lr_linear_plan(8, 8, 8, 0, 0, None) == -1
    for M in (1, 33, 65, 777, 16384):
        for N, K in ((8, 8), (1280, 8192), (28672, 4096), (4096, 14336)):
            for pair in (False, True):
                for scratch in (0, 1 << 20, 64 << 20):
                    p = _hip.linear_plan(M, N, K, pair, scratch)
                    assert p.whole + p.cut == -(-M // p.tile_rows) * -(-N // p.tile_cols)
                    assert p.sums_bytes == p.cut * p.pieces * p.tile_rows * p.tile_cols * 4 <= scratch
                    assert (p.pieces == 1) == (p.cut == 0) and p.pieces <= -(-K // 128)


def test_products_with_memory_for_partial_sums_refuse_what_the_ones_without_refuse(lib):
    """Only refusals: nothing here may reach a launch."""
    from gpt_fast._hip import _RopeKv

    E_NULL, E_ALIGN, E_SHAPE = -1, -2, -3
    p = 4096
    rope = _RopeKv(p, p, p, p, None, 8, 1, 128, 64, 64)      # N = (8 + 2) * 128 = 1280

    def linear(x=p, ldx=64, w=p, y=p, ldy=48, M=40, N=48, K=64, scratch=p):
        return lib.lr_linear_scratch(x, ldx, w, y, ldy, M, N, K, scratch, 1 << 20, None)

    def fused(x=p, ldx=64, y=p, ldy=1280, M=40, K=64, S=1, r=rope, scratch=p):
        return lib.lr_linear_rope_kv_scratch(x, ldx, p, y, ldy, M, K, S, None if r is None else ctypes.byref(r), scratch, 1 << 20, None)

    def swiglu(x=p, ldx=64, y=p, ldy=24, M=40, N=48, K=64, scratch=None, sums=p):
        return lib.lr_linear_swiglu_out_scratch(x, ldx, p, y, ldy, M, N, K, scratch, 0, sums, 1 << 20, None)

    for call in (linear, fused, swiglu):
        assert call(x=None) == E_NULL and call(y=None) == E_NULL
        assert call(x=p + 8) == E_ALIGN and call(y=p + 2) == E_ALIGN
        assert call(M=0) == E_SHAPE and call(K=0) == E_SHAPE and call(ldx=56) == E_SHAPE and call(ldy=16) == E_SHAPE
        assert call(K=60) == E_ALIGN and call(ldx=68) == E_ALIGN
    assert linear(w=None) == E_NULL and linear(scratch=p + 8) == E_ALIGN and fused(scratch=p + 8) == E_ALIGN
    assert swiglu(sums=p + 8) == E_ALIGN and swiglu(N=47) == E_SHAPE
    assert fused(r=None) == E_NULL and fused(M=41, S=2) == E_SHAPE and fused(ldy=1284) == E_ALIGN
    # the projection's buffer may be missing for up to 64 rows and for large grids, not in between
    for M, N in ((65, 48), (511, 1 << 16), (1536, 7936)):      # (186 tiles of 256 rows x 128 pairs)
        assert swiglu(M=M, N=N, ldy=N // 2) == E_NULL


def test_linear_resid_refuses_what_it_cannot_serve(lib):
    """Checked before anything is launched: missing parts, more rows than its bands hold, misaligned rows."""
    from gpt_fast import _hip

    def rc(M=4, **kw):
        d = _hip._LinearResid(**{**dict(x1=256, w1=256, x2=256, w2=256, ldx1=64, ldx2=64, K1=64, K2=64, D=64, resid_in=256, resid_out=256,
                                        gain1=256, gain2=256, out1=256, out2=256, sums1=256, sums2=256), **kw})
        return lib.lr_linear_resid(ctypes.byref(d), M, None)

    assert lib.lr_linear_resid(None, 4, None) == -1
    for name in ("x1", "w1", "x2", "w2", "gain1", "gain2", "out1", "out2", "sums1", "sums2", "resid_in", "resid_out"):
        assert rc(**{name: None}) == -1, name
    assert rc(joint=1, gain2=None) == -1 and rc(M=0) == -3 and rc(M=17) == -4
    assert rc(K1=60) == -2 and rc(ldx2=60) == -3 and rc(w1=250) == -2


@pytest.mark.parametrize("entry", ["linear_multi", "linear_fp8_multi", "attn_decode_beside", "attn_decode_beside_fp8"])
def test_undivided_rows_are_refused_where_they_cannot_be_served(lib, entry):
    """Checked before anything is launched: sums of another width than the rows, more parts or rows than a launch holds, a total
    with no place to go."""
    from gpt_fast import _hip

    fp8 = "fp8" in entry
    q = (_hip._ProjectionFp8 if fp8 else _hip._Projection)()
    q.x, q.ldx, q.y, q.ldy, q.N, q.K, q.epilogue = 256, 64, 256, 64, 64, 64, _hip.EPI_NONE
    if fp8:
        q.w8, q.scales = 256, 256
    else:
        q.w = 256

    def rc(M=4, **kw):
        norm = _hip._RowNorm(**{**dict(sums=256, count=2, dim=64, eps=1e-5), **kw})
        p, n = ctypes.cast(ctypes.byref(q), ctypes.c_void_p), ctypes.byref(norm)
        if "beside" in entry:
            return getattr(lib, f"lr_{entry}_normed")(256, 256, 256, 256, 256, 256, 256, M, 2, 1, 64, 64, 256, 1 << 20, p, n, M, None)
        return getattr(lib, f"lr_{entry}_normed")(p, n, 1, M, None)

    assert rc(count=0) == -3 and rc(dim=72) == -3 and rc(count=513) == -4 and rc(sums=264) == -2
    assert rc(fold_sums=256, fold_count=2) == -1 and rc(fold_sums=264, fold_total=256, fold_count=2) == -2
    assert rc(fold_sums=256, fold_total=256, fold_count=0) == -3 and rc(fold_sums=256, fold_total=256, fold_count=513) == -4
    assert rc(M=17) == -4
    if fp8:
        assert rc(M=1) == -4      # (one row: the matrix-vector kernel)


def test_ladder_block_and_pieces_refuse_what_they_cannot_serve(lib):
    """Checked before anything is launched."""
    from gpt_fast import _hip

    pointers = ("x", "xn", "xn2", "qkv", "y", "act", "h", "a", "m", "gain1", "gain2", "wqkv", "wo", "w1", "w2")
    heads = dict(n_head=4, n_kv_head=2, head_dim=64, smax=64, block_size=64)

    def rc(rope=None, **kw):
        r = _hip._RopeKv(**{**dict(table=256, pos=256, k_cache=256, v_cache=256), **heads, **(rope or {})})
        d = _hip._LadderBlock(**{**{n: 256 for n in pointers}, **dict(B=1, S=8, dim=64, ffn=64, eps=1e-5, rope=r, a_pieces=-1, m_pieces=-1), **kw})
        return lib.lr_ladder_block(ctypes.byref(d), None)

    assert lib.lr_ladder_block(None, None) == -1
    for name in pointers:
        assert rc(**{name: None}) == -1 and rc(**{name: 264}) == -2, name
    for name in ("table", "pos", "k_cache", "v_cache"):
        assert rc(rope={name: None}) == -1, name
    for name in heads:
        assert rc(rope={name: 0}) == -3, name
    assert rc(rope=dict(n_head=5)) == -3 and rc(rope=dict(head_dim=60)) == -2
    assert rc(S=4) == -4 and rc(S=0) == -3 and rc(dim=60) == -2 and rc(ffn=60) == -2 and rc(a_pieces=2) == -1 and rc(sums_a=8) == -2

    n = ctypes.c_int32()
    pieces = lambda x=256, ldx=64, w=256, M=64, N=64, K=64, sums=256, size=1 << 20, out=ctypes.byref(n): \
        lib.lr_linear_pieces(x, ldx, w, M, N, K, sums, size, out, None)
    for name in ("x", "w", "sums", "out"):
        assert pieces(**{name: None}) == -1, name
    assert pieces(K=60) == -2 and pieces(ldx=56) == -3 and pieces(N=0) == -3
    assert pieces(M=32) == -4 and pieces(N=66) == -4 and pieces(size=64) == -4      # nothing is cut
    norms = lambda d1=256, p1=0, d2=256, p2=0: lib.lr_ladder_norms_pieces(256, d1, p1, d2, p2, 256, 256, 256, 256, 256, 8, 60, 1e-5, None)
    assert norms(p1=-1) == -3 and norms(d1=None, p1=2) == -1 and norms(d2=None, p2=2) == -1 and norms(p1=2, p2=3) == -2


def test_two_products_of_one_launch_refuse_what_they_cannot_serve(lib):
    """Memory that both would write among it; what two launches serve is declined."""
    n0, n1 = ctypes.c_int32(), ctypes.c_int32()

    def two(x0=256, w0=256, K0=1024, sums0=1 << 30, n0=ctypes.byref(n0), x1=256, w1=256, K1=1024, sums1=2 << 30, n1=ctypes.byref(n1), M=64, N=64,
            size=1 << 20):
        return lib.lr_linear_pieces_two(x0, w0, K0, sums0, n0, x1, w1, K1, sums1, n1, M, N, size, None)

    for name in ("x0", "w0", "sums0", "n0", "x1", "w1", "sums1", "n1"):
        assert two(**{name: None}) == -1, name
    for name in ("x0", "w0", "sums0", "x1", "w1", "sums1"):
        assert two(**{name: 264}) == -2, name
    for name in ("M", "N", "K0", "K1"):
        assert two(**{name: 0}) == -3, name
    assert two(K0=1028) == -2 and two(K1=1028) == -2
    assert two(sums1=1 << 30) == -3 and two(sums1=(1 << 30) + (1 << 20) - 256) == -3 and two(sums1=(1 << 30) - 256) == -3
    assert two(M=16) == -4 and two(N=66) == -4 and two(K0=1032) == -4 and two(size=0) == -4
    assert lib.lr_linear_pieces_two_bytes(16, 64, 1024, 1024) == 0 == lib.lr_linear_pieces_two_bytes(64, 66, 1024, 1024)
    assert lib.lr_linear_pieces_two_bytes(64, 0, 1024, 1024) == 0 == lib.lr_linear_pieces_two_bytes(64, 64, 1028, 1024)


def test_linear_residual_rms_refuses_what_it_cannot_serve(lib):
    """Checked before anything is launched; memory that some bands would write while others read it among it."""
    from gpt_fast import _hip

    at = {n: (i + 1) << 24 for i, n in enumerate(("x", "w", "resid", "gain_before", "gain", "x_compute", "sums", "parts"))}

    def rc(M=4, N=32768, K=64, ldx=64, before=True, norm={}, **kw):   # (wider than any rows that are served: nothing reaches a launch)
        p = {**at, **kw}
        b = _hip._RowNorm(**{**dict(sums=p["parts"], count=32, dim=N, eps=1e-5), **norm})
        return lib.lr_linear_residual_rms(p["x"], ldx, p["w"], M, N, K, p["resid"], 1.0, ctypes.byref(b) if before else None, p["gain_before"], p["gain"],
                                          1.0, p["x_compute"], p["sums"], None)

    for name in ("x", "w", "resid", "gain_before", "gain", "x_compute", "sums", "parts"):
        assert rc(**{name: None}) == -1, name
    for name in ("x", "w", "resid", "gain_before", "gain", "x_compute"):
        assert rc(**{name: at[name] + 8}) == -2, name
    assert rc(M=0) == -3 and rc(N=0) == -3 and rc(K=0) == -3 and rc(K=60) == -2 and rc(ldx=56) == -3 and rc(M=17) == -4
    assert rc(norm=dict(dim=64)) == -3 and rc(norm=dict(fold_sums=256)) == -3
    ranges = dict(x=(3 * 64 + 64) * 2, resid=4 * 32768 * 4, x_compute=4 * 32768 * 2, sums=16, gain=65536, gain_before=65536, parts=4 * 32 * 4)
    for out in ("resid", "x_compute", "sums"):
        for other in ranges:
            if other != out:
                assert rc(**{out: at[other]}) == -3, (out, other)                              # the same place
                assert rc(**{out: at[other] + ranges[other] - 16}) == -3, (out, other)         # its last 16 bytes
                assert rc(**{other: at[out] + ranges[out] - 16}) == -3, (out, other)
                assert rc(**{out: at[other] - ranges[out]}) == -4, (out, other)                # next to it
    assert rc(before=False, sums=at["parts"], gain_before=None) == -4


def test_products_on_e4m3_weights_refuse_what_they_cannot_serve(lib):
    """Checked before anything is launched; shapes of the passes of 16 rows are declined."""
    from gpt_fast import _hip

    heads = dict(n_head=4, n_kv_head=2, head_dim=64, smax=64, block_size=64)

    def one(x=256, ldx=128, w=256, scales=256, y=256, ldy=512, M=17, N=512, K=128, sums=256, size=0, rope=None):
        r = None if rope is None else ctypes.byref(_hip._RopeKv(**{**dict(table=256, pos=256, k_cache=256, v_cache=256), **heads, **rope}))
        return lib.lr_linear_fp8_product(x, ldx, w, scales, y, ldy, M, N, K, r, sums, size, None)

    for name in ("x", "w", "scales", "y"):
        assert one(**{name: None}) == -1, name
    for name in ("x", "w", "y", "sums"):
        assert one(**{name: 264}) == -2, name
    assert one(M=0) == -3 and one(N=0) == -3 and one(K=0) == -3 and one(ldx=120) == -3 and one(ldy=504) == -3 and one(K=120) == -2 and one(ldx=132) == -2
    assert one(M=16) == -4 and one(M=65) == -4 and one(K=64) == -4 and one(K=192, ldx=192) == -4
    for name in ("table", "pos", "k_cache", "v_cache"):
        assert one(rope={name: None}) == -1, name
    for name in heads:
        assert one(rope={name: 0}) == -3, name
    assert one(rope=dict(n_head=5)) == -3

    n0, n1 = ctypes.c_int32(), ctypes.c_int32()

    def two(x0=256, w0=256, s0=256, K0=1024, sums0=1 << 30, n0=ctypes.byref(n0), x1=256, w1=256, s1=256, K1=1024, sums1=2 << 30, n1=ctypes.byref(n1),
            M=64, N=64, size=1 << 20):
        return lib.lr_linear_fp8_pieces_two(x0, w0, s0, K0, sums0, n0, x1, w1, s1, K1, sums1, n1, M, N, size, None)

    for name in ("x0", "w0", "s0", "sums0", "n0", "x1", "w1", "s1", "sums1", "n1"):
        assert two(**{name: None}) == -1, name
    for name in ("x0", "w0", "sums0", "x1", "w1", "sums1"):
        assert two(**{name: 264}) == -2, name
    for name in ("M", "N", "K0", "K1"):
        assert two(**{name: 0}) == -3, name
    assert two(K0=1032) == -2 and two(sums1=1 << 30) == -3 and two(sums1=(1 << 30) + (1 << 20) - 256) == -3
    assert two(M=16) == -4 and two(M=65) == -4 and two(N=66) == -4 and two(K0=1040) == -4 and two(size=0) == -4
    assert lib.lr_linear_fp8_pieces_two_bytes(16, 64, 1024, 1024) == 0 == lib.lr_linear_fp8_pieces_two_bytes(64, 66, 1024, 1024)
    assert lib.lr_linear_fp8_product_bytes(16, 512, 128, 0) == 0 == lib.lr_linear_fp8_product_bytes(64, 511, 128, 1)

    def beside(scales=256, x=256, w=256, act=256, M=17, N=512, K=128, ldx=128, ldact=256, sums=256, q=256, Hq=8):
        return lib.lr_attn_decode_beside_product_fp8(q, 1024, 256, 256, 256, 256, 1024, 32, Hq, 1, 128, 64, 256, 1 << 24, 256, x, ldx, w, scales, act, ldact, M,
                                                     N, K, sums, 1 << 20, None)

    for name in ("scales", "x", "w", "act", "q"):
        assert beside(**{name: None}) == -1, name
    assert beside(x=264) == -2 and beside(sums=264) == -2 and beside(N=511) == -3 and beside(ldx=120) == -3 and beside(ldact=248) == -3 and beside(Hq=0) == -3
    assert beside(M=16) == -4 and beside(M=65) == -4 and beside(K=64) == -4


def test_add_rmsnorm_of_partial_sums_refuses_what_it_cannot_serve(lib):
    def rc(resid=256, d1=256, pieces=2, d2=None, gain=256, out=256, normed=256, rows=4, dim=64):
        return lib.lr_add_rmsnorm_pieces(resid, d1, pieces, d2, gain, out, normed, rows, dim, 1e-5, None)

    assert rc(d1=None) == -1 and rc(resid=None) == -1 and rc(gain=None) == -1 and rc(normed=None) == -1 and rc(pieces=-1) == -3
    assert rc(d1=264) == -2 and rc(d2=264) == -2 and rc(dim=60) == -2 and rc(rows=0) == -3 and rc(dim=32768) == -4


@pytest.mark.parametrize("entry", ["beside_merged", "beside_fp8_merged", "beside_product"])
def test_attention_in_a_shared_launch_refuses_what_its_own_launch_refuses(lib, entry):
    """lr_attn_decode's arguments and the tickets; what is not for these grids is declined."""
    from gpt_fast import _hip

    proj = _hip._ProjectionFp8 if "fp8" in entry else _hip._Projection
    p = proj(**{**{"w8" if "fp8" in entry else "w": 256}, **dict(x=256, y=256, ldx=64, ldy=64, N=64, K=64, epilogue=0), **(dict(scales=256) if "fp8" in entry else {})})

    def rc(q=256, ldq=1024, k=256, v=256, pos=256, y=256, ldy=1024, B=32, Hq=8, Hkv=1, hd=128, Smax=64, scratch=256, n=1 << 24, tickets=256, M=16,
           K=64):
        a = q, ldq, k, v, pos, y, ldy, B, Hq, Hkv, hd, Smax, scratch, n
        if entry == "beside_product":
            return lib.lr_attn_decode_beside_product(*a, tickets, 256, 64, 256, 256, 64, 2 * M, 128, K, 256, 1 << 20, None)
        return getattr(lib, "lr_attn_decode_" + entry)(*a, ctypes.cast(ctypes.byref(p), ctypes.c_void_p), None, tickets, M, None)

    for name in ("q", "k", "v", "y", "scratch", "pos"):
        assert rc(**{name: None}) == -1, name
    for name in ("q", "k", "v", "y", "scratch"):
        assert rc(**{name: 264}) == -2, name
    for name in ("B", "Hq", "Hkv", "hd", "Smax", "M"):
        assert rc(**{name: 0}) == -3, name
    assert rc(ldq=1016) == -3 and rc(ldy=1016) == -3 and rc(ldq=1028) == -2 and rc(ldy=1028) == -2 and rc(Hkv=3) == -3 and rc(n=16) == -3
    assert rc(B=65536) == -3 and rc(tickets=258) == -2
    assert rc(M=33) == -4 and rc(Hq=3, Hkv=1) == -4 and rc(hd=96) == -4
    if entry == "beside_product":
        assert rc(tickets=None) == -1 and rc(K=4) == -2 and rc(K=72, M=16) == -3 and rc(Smax=17000, n=1 << 30) == -4 and rc(M=8) == -4
        assert lib.lr_attn_decode_beside_product(256, 1024, 256, 256, 256, 256, 1024, 32, 8, 1, 128, 64, 256, 1 << 24, 256, 256, 64, 256, 256, 63, 32,
                                                 128, 64, 256, 1 << 20, None) == -3      # rows of the activation
        return
    assert rc(M=17) == -4
    null = getattr(lib, "lr_attn_decode_" + entry)(256, 1024, 256, 256, 256, 256, 1024, 4, 8, 1, 128, 64, 256, 1 << 24, None, None, 256, 4, None)
    assert null == -1


def test_expanded_weights_of_a_graph_are_in_memory_of_its_own(lib, monkeypatch):
    """Of calls on one stream the eager ones share a buffer that grows; what is captured neither takes nor leaves one there."""
    from types import SimpleNamespace

    from gpt_fast import _hip

    made, capturing = [], [False]
    monkeypatch.setattr(_hip, "_FP8_SCRATCH", {})
    monkeypatch.setattr(_hip, "_stream", lambda: 7)
    monkeypatch.setattr(_hip.torch, "empty", lambda n, **kw: made.append(n) or SimpleNamespace(numel=lambda: n))
    monkeypatch.setattr(_hip.torch.cuda, "is_current_stream_capturing", lambda: capturing[0])
    dev = torch.device("cuda", 0)
    a = _hip._fp8_scratch(dev, 100)
    assert _hip._fp8_scratch(dev, 50) is a
    capturing[0] = True
    g = [_hip._fp8_scratch(dev, n) for n in (50, 50, 200)]
    assert a not in g and g[0] is not g[1] and list(_hip._FP8_SCRATCH.values()) == [a]
    capturing[0] = False
    assert _hip._fp8_scratch(dev, 100) is a
    b = _hip._fp8_scratch(dev, 200)
    assert b not in g and made == [100, 50, 50, 200, 200] and _hip._fp8_scratch(dev, 200) is b


def test_ladder_block_refuses_more_partial_sums_than_its_memory_holds(lib):
    """What the block before left is read in whole pieces of rows x dim: a count that the memory cannot hold is a mistake of the
    caller's, found before anything is launched."""
    from gpt_fast import _hip

    pointers = ("x", "xn", "xn2", "qkv", "y", "act", "h", "a", "m", "gain1", "gain2", "wqkv", "wo", "w1", "w2", "sums_a", "sums_m")
    r = _hip._RopeKv(table=256, pos=256, k_cache=256, v_cache=256, n_head=4, n_kv_head=2, head_dim=64, smax=64, block_size=64)
    for which in ("a_pieces", "m_pieces"):
        for pieces, size in ((1, 40 * 64 * 4 - 1), (3, 40 * 64 * 4 * 3 - 1), (0x7fffffff, 1 << 26)):
            d = _hip._LadderBlock(**{n: 256 for n in pointers}, B=1, S=40, dim=64, ffn=64, eps=1e-5, rope=r, sums_bytes=size,
                                  **{**dict(a_pieces=-1, m_pieces=-1), which: pieces})
            assert lib.lr_ladder_block(ctypes.byref(d), None) == -3, (which, pieces)


def test_a_profile_builds_stamps_stay_in_the_buffer_it_asks_for(tmp_path):
    """Host part of the bands' sources, as a profile build compiles them: the last stamp of a workgroup of any width is its own, and
    the buffer that lr_band_profile asks for ends behind the last one."""
    import shutil
    import subprocess

    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    csrc = os.path.join(ROOT, "ladder-residual-inference_amd", "csrc")
    src = tmp_path / "stamps.hip"
    src.write_text(f'''#define LR_BAND_PROFILE
#include "{csrc}/stream_gemm.hip"
static_assert(band_prof_at(3, RN_WAVES - 1, 5) < band_prof_at(4, 0, 0) && band_prof_at(3, NWV - 1, 5) < band_prof_at(4, 0, 0), "");
static_assert(band_prof_bytes(4) >= (long long)sizeof(unsigned long long) * (band_prof_at(3, RN_WAVES - 1, 5) + 1), "");
''')
    r = subprocess.run([hipcc, "--cuda-host-only", "-fsyntax-only", "-std=c++17", "-x", "hip", "--offload-arch=gfx950", str(src)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
