"""Per-kernel parity on a real MI355X: every C-ABI entry point of libladder_hip.so against the
oracle's op (oracle/ladder_oracle.py, eager PyTorch on the same device, same seeded inputs).

Tolerances, all stated in bf16 units-in-the-last-place ("ulp") of the produced tensor:
  * pure data movement and element-wise work with one rounding (embed, add, RoPE, cache write,
    argmax, advance): bit-exact;
  * ops with an fp32 reduction inside (RMSNorm, linear, attention) or a transcendental (SwiGLU):
    the fp32 value before the final rounding differs from the oracle's by summation order /
    libm only, so results must agree within 1 ulp and on all but a small fraction of elements."""
import math

import pytest
import torch
import torch.nn.functional as F

from oracle import ladder_oracle as O

pytestmark = pytest.mark.gpu

DEV = "cuda"
BF = torch.bfloat16


@pytest.fixture(scope="module")
def hip():
    from gpt_fast import _hip

    _hip.load()
    return _hip


def rnd(*shape, seed=0, scale=1.0, dtype=BF):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return (torch.randn(*shape, generator=g, device=DEV) * scale).to(dtype)


def ulp_diff(a: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    """Distance in bf16 steps between two bf16 tensors (monotonic integer mapping of the bits)."""
    def key(t):
        i = t.contiguous().view(torch.int16).to(torch.int32)
        return torch.where(i < 0, -(i & 0x7FFF), i)
    return (key(a) - key(b)).abs()


def assert_close_ulp(got, want, max_ulp=1, max_frac=0.02, what=""):
    assert got.shape == want.shape and got.dtype == want.dtype == BF
    assert torch.isfinite(got.float()).all(), what
    d = ulp_diff(got, want)
    # values whose magnitude is far below the tensor's scale may differ by many ulps of their own
    # size while being equal to fp32 accuracy relative to the sum that produced them
    tiny = want.float().abs() < want.float().abs().max() * 2.0 ** -12
    bad = (d > max_ulp) & ~tiny
    frac = (d > 0).float().mean().item()
    assert not bad.any(), f"{what}: {int(bad.sum())} elements differ by more than {max_ulp} ulp (max {int(d.max())})"
    assert frac <= max_frac, f"{what}: {frac:.4f} of elements differ (limit {max_frac})"


# ------------------------------------------------------------------------------------ embed / add / advance

@pytest.mark.parametrize("idx_dtype", [torch.int64, torch.int32])
def test_embed_exact(hip, idx_dtype):
    table = rnd(1000, 512, seed=1)
    idx = torch.randint(0, 1000, (3, 17), device=DEV, dtype=idx_dtype)
    out = torch.empty(3 * 17, 512, dtype=BF, device=DEV)
    hip.embed(table, idx, out)
    assert torch.equal(out.view(3, 17, 512), F.embedding(idx.long(), table))


@pytest.mark.parametrize("n", [8, 2048, 8192 * 5 + 24, 1000003])
def test_add_exact(hip, n):
    a, b = rnd(n, seed=2), rnd(n, seed=3)
    out = torch.empty_like(a)
    hip.add(a, b, out)
    assert torch.equal(out, a + b)
    hip.add(a, b, out, b_div=8.0)
    assert torch.equal(out, a + b / 8)
    hip.add(a, b, out, b_div=3.0)
    assert torch.equal(out, a + b / 3)
    out2 = b.clone()
    hip.add(a, out2, out2)  # aliasing the second operand
    assert torch.equal(out2, a + b)


def test_advance_and_history(hip):
    B = 5
    cur = torch.zeros(B, 1, dtype=torch.int32, device=DEV)
    nxt = torch.arange(10, 10 + B, dtype=torch.int32, device=DEV).view(B, 1)
    pos = torch.tensor([7], dtype=torch.int32, device=DEV)
    hist = torch.full((B, 4), -1, dtype=torch.int32, device=DEV)
    hip.advance(cur, nxt, pos, B, hist, pos0=6)
    assert pos.item() == 8 and torch.equal(cur, nxt) and hist[:, 1].tolist() == list(range(10, 10 + B))
    assert (hist[:, [0, 2, 3]] == -1).all()
    hip.advance(None, None, pos, B)
    assert pos.item() == 9


# ------------------------------------------------------------------------------------ RMSNorm

@pytest.mark.parametrize("rows,dim", [(1, 8192), (3, 4096), (64, 8192), (2, 16384), (5, 256), (2048, 2048)])
def test_add_rmsnorm(hip, rows, dim):
    r, d1, d2 = rnd(rows, dim, seed=4), rnd(rows, dim, seed=5, scale=0.1), rnd(rows, dim, seed=6, scale=0.1)
    g = rnd(dim, seed=7, scale=0.02)
    ro, no = torch.empty_like(r), torch.empty_like(r)
    # plain norm
    hip.add_rmsnorm(r, None, None, g, None, no, 1e-5)
    # two roundings in a row (normalised value, then gain product): a 1-ulp flip of the first can
    # show as 2 ulp after the second, hence max_ulp=2 for this op only
    assert_close_ulp(no, O.rms_norm(r, g, 1e-5), max_ulp=2, max_frac=0.01, what="norm")
    # one pending partial (ladder add), residual written back
    hip.add_rmsnorm(r, d1, None, g, ro, no, 1e-5)
    assert torch.equal(ro, r + d1)
    assert_close_ulp(no, O.rms_norm(r + d1, g, 1e-5), max_ulp=2, max_frac=0.01, what="add+norm")
    # two pending partials (closing add of the ladder), in place
    r2 = r.clone()
    hip.add_rmsnorm(r2, d1, d2, g, r2, no, 1e-5)
    assert torch.equal(r2, r + d1 + d2)
    assert_close_ulp(no, O.rms_norm(r + d1 + d2, g, 1e-5), max_ulp=2, max_frac=0.01, what="add+add+norm")


# ------------------------------------------------------------------------------------ linear

def linear_ref(x, w):
    """fp64 product rounded once: what any fp32-accumulating bf16 linear must match within 1 ulp."""
    return (x.double() @ w.double().T).to(BF)


GEMV_SHAPES = [  # (N, K): the 70B rank shard, the 8B model, the 1B model, and ragged sizes
    (1280, 8192), (8192, 1024), (7168, 8192), (8192, 3584), (16032, 8192),
    (6144, 4096), (4096, 4096), (3072, 2048), (2048, 8192), (24, 64), (1001, 520),
]


@pytest.mark.parametrize("N,K", GEMV_SHAPES)
@pytest.mark.parametrize("M", [1, 2, 3, 5, 8])
def test_linear_gemv(hip, M, N, K):
    x = rnd(M, K, seed=8)
    w = rnd(N, K, seed=9, scale=0.02)
    y = torch.empty(M, N, dtype=BF, device=DEV)
    hip.linear(x, w, y)
    assert_close_ulp(y, linear_ref(x, w), what=f"gemv M={M} N={N} K={K}")
    # and against the library routine the reference uses
    assert_close_ulp(y, F.linear(x, w), max_frac=0.05, what="gemv vs F.linear")


@pytest.mark.parametrize("N,K", [(1280, 8192), (8192, 1024), (7168, 8192), (8192, 3584), (16032, 8192), (4096, 4096),
                                 (4096, 14336), (24, 64), (1001, 520), (130, 136), (33, 8)])
@pytest.mark.parametrize("M", [5, 8, 16, 17, 31, 33, 64])
def test_linear_decode_batches(hip, M, N, K):
    """Decode batches (4 < M <= 64) take the weight-streaming matrix-core kernel: ragged N (bands that end
    inside a 16-row unit), K not a multiple of the 128-element chunk or shorter than one, M on both sides
    of the 16-row column tiles, a strided output view."""
    x = rnd(M, K, seed=12)
    w = rnd(N, K, seed=13, scale=0.02)
    y = torch.empty(M, N, dtype=BF, device=DEV)
    hip.linear(x, w, y)
    assert_close_ulp(y, linear_ref(x, w), what=f"decode batch M={M} N={N} K={K}")
    if N % 8 == 0:
        wide = torch.zeros(M, N + 8, dtype=BF, device=DEV)
        hip.linear(x, w, wide[:, :N])
        assert torch.equal(wide[:, :N], y) and bool((wide[:, N:] == 0).all())


def swiglu_of_projection_ref(x, w1):
    """[up; gate] rows -> bf16(bf16(silu(g)) * u) with u, g the projections rounded to bf16 (utils.py:145-148)."""
    h = linear_ref(x, w1)
    inter = w1.shape[0] // 2
    return F.silu(h[:, inter:]) * h[:, :inter]   # feed_forward of the oracle: silu(g) * u on bf16 tensors


@pytest.mark.parametrize("M,D,NQ,I", [(8, 8192, 1280, 3584), (64, 8192, 1280, 3584), (16, 4096, 6144, 14336),
                                      (5, 264, 40, 50), (33, 136, 520, 17), (1, 512, 96, 200), (64, 72, 8, 1000)])
def test_linear_multi_two_projections_one_launch(hip, M, D, NQ, I):
    """q/k/v projection next to the up/gate projection with the SwiGLU epilogue, in one launch: each output
    against the oracle's op on its own input; bands of different heights in the two projections."""
    xa, xb = rnd(M, D, seed=30), rnd(M, D, seed=31)
    wq, w1 = rnd(NQ, D, seed=32, scale=0.03), rnd(2 * I, D, seed=33, scale=0.03)
    q = torch.empty(M, NQ, dtype=BF, device=DEV)
    act = torch.full((M, I), 3.0, dtype=BF, device=DEV)
    hip.linear_multi((xa, wq, q, hip.EPI_NONE), (xb, w1, act, hip.EPI_SWIGLU))
    assert_close_ulp(q, linear_ref(xa, wq), what="multi: plain projection")
    # u and g may each sit one ulp away from the fp64-rounded projections; the activation amplifies that
    want = swiglu_of_projection_ref(xb, w1)
    assert torch.isfinite(act.float()).all()
    err = (act.float() - want.float()).abs().max().item()
    assert err <= 2.0 ** -6 * want.float().abs().max().item(), err
    assert (ulp_diff(act, want) > 1).float().mean().item() < 0.05
    # the same projections one at a time give the same bits
    q1, act1 = torch.empty_like(q), torch.empty_like(act)
    hip.linear_multi((xa, wq, q1, hip.EPI_NONE))
    hip.linear_multi((xb, w1, act1, hip.EPI_SWIGLU))
    assert torch.equal(q1, q) and torch.equal(act1, act)


def test_linear_multi_swiglu_epilogue_equals_the_two_step_path(hip):
    """The fused epilogue rounds where the unfused path rounds: w1 -> h (bf16) -> lr_swiglu gives the same bits."""
    M, D, I = 8, 1024, 520
    x, w1 = rnd(M, D, seed=34), rnd(2 * I, D, seed=35, scale=0.03)
    act = torch.empty(M, I, dtype=BF, device=DEV)
    hip.linear_multi((x, w1, act, hip.EPI_SWIGLU))
    h = torch.empty(M, 2 * I, dtype=BF, device=DEV)
    hip.linear_multi((x, w1, h, hip.EPI_NONE))
    two_step = torch.empty(M, I, dtype=BF, device=DEV)
    hip.swiglu(h, two_step)
    assert torch.equal(act, two_step)


@pytest.mark.parametrize("B,Hq,Hkv,hd,D", [(8, 8, 1, 128, 1024), (64, 8, 1, 128, 512), (16, 32, 8, 128, 264),
                                            (5, 4, 2, 64, 136), (1, 2, 2, 64, 64)])
@pytest.mark.parametrize("pos_value", [0, 37])
def test_linear_multi_rope_kv_epilogue_equals_projection_then_rope_kv_write(hip, B, Hq, Hkv, hd, D, pos_value):
    """The q/k/v projection that rotates and caches on its way out leaves q, the K slot and the V slot exactly as
    the plain projection followed by lr_rope_kv_write does, and touches no other cache slot."""
    Smax, block = 48, 64
    N = (Hq + 2 * Hkv) * hd
    x, w = rnd(B, D, seed=40), rnd(N, D, seed=41, scale=0.05)
    table = O.rope_table(block, hd, 10000.0, BF).to(DEV)
    pos = torch.tensor([pos_value], dtype=torch.int32, device=DEV)
    kc = [rnd(B, Hkv, Smax, hd, seed=42) for _ in range(2)]
    vc = [rnd(B, Hkv, Smax, hd, seed=43) for _ in range(2)]
    # reference path
    q_ref = torch.empty(B, N, dtype=BF, device=DEV)
    hip.linear_multi((x, w, q_ref, hip.EPI_NONE))
    k_proj = q_ref[:, Hq * hd:].clone()
    hip.rope_kv_write(q_ref, table, False, pos, kc[0], vc[0], B, 1, Hq, Hkv, hd)
    # fused path
    q = torch.empty(B, N, dtype=BF, device=DEV)
    hip.linear_multi((x, w, q, hip.rope_kv_epilogue(table, pos, kc[1], vc[1], Hq, Hkv, hd)))
    assert torch.equal(q[:, :Hq * hd], q_ref[:, :Hq * hd])
    assert torch.equal(q[:, Hq * hd:], k_proj)          # k and v stay as projected in the row buffer
    assert torch.equal(kc[1], kc[0]) and torch.equal(vc[1], vc[0])
    assert not torch.equal(kc[1][:, :, pos_value], rnd(B, Hkv, Smax, hd, seed=42)[:, :, pos_value])


def test_linear_multi_rope_kv_epilogue_reports_a_position_outside_the_cache(hip):
    B, Hq, Hkv, hd, D, Smax = 8, 4, 1, 64, 128, 16
    N = (Hq + 2 * Hkv) * hd
    x, w = rnd(B, D, seed=44), rnd(N, D, seed=45, scale=0.05)
    table = O.rope_table(32, hd, 10000.0, BF).to(DEV)
    kc, vc = rnd(B, Hkv, Smax, hd, seed=46), rnd(B, Hkv, Smax, hd, seed=47)
    kc0, vc0 = kc.clone(), vc.clone()
    err = hip.device_error_word(DEV)
    err.zero_()
    plain, q = torch.empty(B, N, dtype=BF, device=DEV), torch.empty(B, N, dtype=BF, device=DEV)
    hip.linear_multi((x, w, plain, hip.EPI_NONE))
    hip.linear_multi((x, w, q, hip.rope_kv_epilogue(table, torch.tensor([Smax], dtype=torch.int32, device=DEV), kc, vc,
                                                    Hq, Hkv, hd)))
    torch.cuda.synchronize()
    assert int(err.item()) == hip.DEV_POS_RANGE
    err.zero_()
    assert torch.equal(q, plain) and torch.equal(kc, kc0) and torch.equal(vc, vc0)


@pytest.mark.parametrize("M,D,I", [(5, 264, 56), (64, 1024, 520), (100, 520, 136), (512, 4096, 14336 // 4), (700, 328, 1000),
                                   (2048, 1024, 3584), (2300, 520, 3000), (2300, 512, 3000)])
def test_linear_swiglu_out_equals_projection_then_swiglu(hip, M, D, I):
    """The first MLP projection with the activation in its epilogue -- the streaming kernel's row pairs (M <= 64), the
    256 x 256 tile GEMM on tiles of 128 pairs (M >= 512, ragged edges included), the two-step fallback in between --
    against the oracle's ops, and bit for bit against lr_linear followed by lr_swiglu."""
    x, w1 = rnd(M, D, seed=50), rnd(2 * I, D, seed=51, scale=0.03)
    act = torch.full((M, I), 3.0, dtype=BF, device=DEV)
    scratch = torch.empty(M, 2 * I, dtype=BF, device=DEV)
    hip.linear_swiglu_out(x, w1, act, scratch)
    h = torch.empty(M, 2 * I, dtype=BF, device=DEV)
    hip.linear(x, w1, h)
    two_step = torch.empty(M, I, dtype=BF, device=DEV)
    hip.swiglu(h, two_step)
    want = swiglu_of_projection_ref(x, w1)
    assert torch.isfinite(act.float()).all()
    assert (act.float() - want.float()).abs().max().item() <= 2.0 ** -6 * want.float().abs().max().item()
    assert (ulp_diff(act, want) > 1).float().mean().item() < 0.05
    # same kernel family on both sides (same summation order) wherever the fused form exists: identical bits
    assert torch.equal(act, two_step)


def test_linear_multi_is_deterministic(hip):
    x, w = rnd(64, 8192, seed=36), rnd(1280, 8192, seed=37, scale=0.02)
    ys = []
    for _ in range(4):
        y = torch.empty(64, 1280, dtype=BF, device=DEV)
        hip.linear_multi((x, w, y, hip.EPI_NONE))
        ys.append(y)
    assert all(torch.equal(ys[0], t) for t in ys[1:])


@pytest.mark.parametrize("cfg", [144, 212, 222, 242, 244, 412, 422, 442])
def test_linear_gemv_every_launch_configuration(hip, cfg):
    x = rnd(4, 3584, seed=10)
    w = rnd(1030, 3584, seed=11, scale=0.02)
    y = torch.empty(4, 1030, dtype=BF, device=DEV)
    hip.linear(x, w, y, gemv_cfg=cfg)   # lr_linear_tuned: the configuration is an argument of the call
    assert_close_ulp(y, linear_ref(x, w), what=f"gemv cfg {cfg}")


def test_linear_gemv_is_deterministic(hip):
    x = rnd(1, 8192, seed=12)
    w = rnd(1280, 8192, seed=13, scale=0.02)
    ys = []
    for _ in range(5):
        y = torch.empty(1, 1280, dtype=BF, device=DEV)
        hip.linear(x, w, y)
        ys.append(y)
    assert all(torch.equal(ys[0], t) for t in ys[1:])


@pytest.mark.parametrize("M,N,K", [(9, 256, 64), (128, 128, 64), (130, 1280, 8192), (2048, 1280, 1024),
                                   (333, 1001, 520), (64, 16032, 2048), (16, 8192, 3584), (257, 384, 8),
                                   # 256 x 256 tiles (M >= 512): whole tiles, ragged edges in M, N and K, the
                                   # XCD-aware tile order (M / 256 a multiple of 32) and the plain one
                                   (512, 256, 64), (700, 500, 328), (1024, 6144, 4096), (8192, 512, 136),
                                   (8192 + 3, 257, 72),
                                   # enough 256 x 256 tiles for the large-tile kernel (192 and more): whole tiles
                                   # in the plain and in the XCD-aware order, ragged edges in M and N with K a
                                   # multiple of the k-tile (scalar k offsets) and with a K tail (per-lane checks)
                                   (4096, 3072, 1024), (8192, 1536, 512), (5000, 3000, 512), (5000, 3000, 328),
                                   (6144, 2048, 64)])
def test_linear_gemm(hip, M, N, K):
    x = rnd(M, K, seed=14)
    w = rnd(N, K, seed=15, scale=0.02)
    y = torch.empty(M, N, dtype=BF, device=DEV)
    hip.linear(x, w, y)
    assert_close_ulp(y, linear_ref(x, w), what=f"gemm M={M} N={N} K={K}")


def test_linear_strided_rows(hip):
    big = rnd(6, 3 * 512, seed=16)
    x = big[:, 512:1024]                      # row stride 1536
    w = rnd(200, 512, seed=17, scale=0.05)
    out = torch.zeros(6, 2 * 200, dtype=BF, device=DEV)
    y = out[:, 200:]                          # row stride 400
    hip.linear(x, w, y)
    assert_close_ulp(y.contiguous(), linear_ref(x, w), what="strided")
    assert (out[:, :200] == 0).all()


@pytest.mark.parametrize("rows", [1, 4, 8, 40])
def test_swiglu_and_fused_w2(hip, rows):
    I, D = 3584, 1024
    h = rnd(rows, 2 * I, seed=18)
    w2 = rnd(D, I, seed=19, scale=0.02)
    u, g = h.chunk(2, dim=-1)
    act = F.silu(g) * u
    out = torch.empty(rows, I, dtype=BF, device=DEV)
    hip.swiglu(h, out)
    assert_close_ulp(out, act, max_frac=0.002, what="swiglu")
    y = torch.empty(rows, D, dtype=BF, device=DEV)
    hip.linear(h, w2, y, act_swiglu=True)
    assert_close_ulp(y, linear_ref(act, w2), max_frac=0.05, what="w2(silu(g)*u)")


# ------------------------------------------------------------------------------------ RoPE + cache

@pytest.mark.parametrize("hd,Hq,Hkv", [(128, 8, 1), (64, 32, 8), (128, 32, 8)])
@pytest.mark.parametrize("gathered", [False, True])
def test_rope_kv_write_exact(hip, hd, Hq, Hkv, gathered):
    B, S, Smax, block = 2, 9, 32, 64
    width = (Hq + 2 * Hkv) * hd
    qkv = rnd(B, S, width + 16, seed=20)[..., :width]          # padded rows: row stride != width
    pos = torch.tensor([3, 4, 5, 6, 7, 8, 9, 20, 31], dtype=torch.int32, device=DEV)
    table = O.rope_table(block, hd, 500000, BF).to(DEV)
    kc = torch.zeros(B + 1, Hkv, Smax, hd, dtype=BF, device=DEV)
    vc = torch.zeros_like(kc)
    q, k, v = qkv.clone().split([Hq * hd, Hkv * hd, Hkv * hd], dim=-1)
    fc = table[pos.long()]
    q_ref = O.apply_rope(q.reshape(B, S, Hq, hd), fc)
    k_ref = O.apply_rope(k.reshape(B, S, Hkv, hd), fc).transpose(1, 2)
    kc_ref, vc_ref = kc.clone(), vc.clone()
    O.kv_update(kc_ref, vc_ref, pos.long(), k_ref, v.reshape(B, S, Hkv, hd).transpose(1, 2))

    work = qkv  # rotated in place on the strided view
    hip.rope_kv_write(work, fc.contiguous() if gathered else table, gathered, pos, kc, vc, B, S, Hq, Hkv, hd)
    assert torch.equal(work[..., : Hq * hd].reshape(B, S, Hq, hd), q_ref)
    assert torch.equal(kc, kc_ref) and torch.equal(vc, vc_ref)
    assert torch.equal(work[..., Hq * hd:], torch.cat([k, v], -1))   # k and v columns are left as they were


@pytest.mark.parametrize("B,S,Hq,Hkv,hd,K,Smax,start", [
    # the 256 x 256-tile GEMM with the rotation and the cache writes in its output pass: whole tiles; ragged rows,
    # sequences that end inside a tile, K with a tail, positions that do not start at 0; then shapes below that
    # kernel's threshold (the two-call fallback) and a decode-sized one
    (4, 1024, 16, 4, 128, 1024, 1024, 0), (5, 1000, 32, 16, 64, 520, 1072, 37), (9, 300, 16, 4, 128, 256, 512, 100),
    (2, 100, 8, 1, 128, 512, 136, 0), (3, 1, 8, 2, 64, 264, 16, 5),
])
def test_linear_rope_kv_equals_the_two_calls(hip, B, S, Hq, Hkv, hd, K, Smax, start):
    """lr_linear_rope_kv against lr_linear followed by lr_rope_kv_write on the same buffers: the output rows and both
    caches bit for bit; and the separate calls against the oracle (apply_rope, kv_update) as everywhere."""
    N = (Hq + 2 * Hkv) * hd
    x = rnd(B * S, K, seed=80)
    w = rnd(N, K, seed=81, scale=0.05)
    pos = torch.arange(start, start + S, dtype=torch.int32, device=DEV)
    table = O.rope_table(start + S + 3, hd, 500000, BF).to(DEV)
    want = torch.empty(B * S, N, dtype=BF, device=DEV)
    hip.linear(x, w, want)
    proj = want.clone()
    kc_w = torch.zeros(B + 1, Hkv, Smax, hd, dtype=BF, device=DEV)
    vc_w = torch.zeros_like(kc_w)
    hip.rope_kv_write(want, table, False, pos, kc_w, vc_w, B, S, Hq, Hkv, hd)
    fc = table[pos.long()]
    q, k, v = proj.view(B, S, N).split([Hq * hd, Hkv * hd, Hkv * hd], dim=-1)
    assert torch.equal(want.view(B, S, N)[..., : Hq * hd].reshape(B, S, Hq, hd), O.apply_rope(q.reshape(B, S, Hq, hd), fc))
    kc_o, vc_o = torch.zeros_like(kc_w), torch.zeros_like(kc_w)
    O.kv_update(kc_o, vc_o, pos.long(), O.apply_rope(k.reshape(B, S, Hkv, hd), fc).transpose(1, 2),
                v.reshape(B, S, Hkv, hd).transpose(1, 2))
    assert torch.equal(kc_w, kc_o) and torch.equal(vc_w, vc_o)

    got = torch.full((B * S, N), 7.0, dtype=BF, device=DEV)
    kc, vc = torch.zeros_like(kc_w), torch.zeros_like(kc_w)
    hip.linear_rope_kv(x, w, got, table, pos, kc, vc, B, S, Hq, Hkv, hd)
    assert torch.equal(got, want)
    assert torch.equal(kc, kc_w) and torch.equal(vc, vc_w)
    hip.raise_on_device_error(got.device)


def test_linear_rope_kv_position_out_of_range(hip):
    """A position beyond the cache: that row stays as projected, nothing of it reaches the caches, the device error
    word is set (as lr_rope_kv_write does); the other rows are finished as usual."""
    B, S, Hq, Hkv, hd, K, Smax = 4, 1024, 16, 4, 128, 512, 1024
    N = (Hq + 2 * Hkv) * hd
    x, w = rnd(B * S, K, seed=82), rnd(N, K, seed=83, scale=0.05)
    pos = torch.arange(S, dtype=torch.int32, device=DEV)
    pos[700] = Smax + 5
    table = O.rope_table(2048, hd, 500000, BF).to(DEV)
    want = torch.empty(B * S, N, dtype=BF, device=DEV)
    hip.linear(x, w, want)
    kc_w = torch.zeros(B, Hkv, Smax, hd, dtype=BF, device=DEV)
    vc_w = torch.zeros_like(kc_w)
    hip.device_error_word(want.device).zero_()
    hip.rope_kv_write(want, table, False, pos, kc_w, vc_w, B, S, Hq, Hkv, hd)
    assert int(hip.device_error_word(want.device).item()) != 0
    hip.device_error_word(want.device).zero_()
    got = torch.empty_like(want)
    kc, vc = torch.zeros_like(kc_w), torch.zeros_like(kc_w)
    hip.linear_rope_kv(x, w, got, table, pos, kc, vc, B, S, Hq, Hkv, hd)
    torch.cuda.synchronize()
    assert int(hip.device_error_word(want.device).item()) != 0
    hip.device_error_word(want.device).zero_()
    assert torch.equal(got, want) and torch.equal(kc, kc_w) and torch.equal(vc, vc_w)


@pytest.mark.parametrize("hd,H", [(128, 1), (64, 8), (128, 8)])
@pytest.mark.parametrize("layout", ["bhsd", "bshd"])
def test_kv_cache_update_module_method(hd, H, layout):
    """KVCache.update (utils.py:50-59) through lr_kv_update: dense [B, H, S, D] values and the transposed view of a
    [B, S, H, D] tensor (what a caller holds right after splitting a projection), scattered positions, a batch
    smaller than the cache; bit-exact against the oracle's indexed assignment, rows not addressed stay zero."""
    from gpt_fast.utils import KVCache

    B, S, Smax = 2, 7, 40
    pos = torch.tensor([0, 5, 6, 7, 21, 38, 39], device=DEV)          # int64, as torch.arange gives
    if layout == "bhsd":
        k, v = rnd(B, H, S, hd, seed=70), rnd(B, H, S, hd, seed=71)
    else:
        k, v = rnd(B, S, H, hd, seed=70).transpose(1, 2), rnd(B, S, H, hd, seed=71).transpose(1, 2)
    cache = KVCache(B + 1, Smax, H, hd).to(DEV)
    kc_ref, vc_ref = cache.k_cache.clone(), cache.v_cache.clone()
    O.kv_update(kc_ref, vc_ref, pos, k, v)
    k_out, v_out = cache.update(pos, k, v)
    assert k_out is cache.k_cache and v_out is cache.v_cache
    assert torch.equal(k_out, kc_ref) and torch.equal(v_out, vc_ref)
    assert float(k_out[B].abs().max()) == 0.0 and float(k_out[:, :, 1].abs().max()) == 0.0


def test_kv_cache_update_reports_a_position_outside_the_cache(hip):
    from gpt_fast.utils import KVCache

    cache = KVCache(1, 16, 2, 64).to(DEV)
    k = rnd(1, 2, 2, 64, seed=72)
    hip.device_error_word(DEV).zero_()
    cache.update(torch.tensor([3, 16], device=DEV), k, k)
    torch.cuda.synchronize()
    assert int(hip.device_error_word(DEV).item()) == 2            # LR_DEV_POS_RANGE; slot 3 was still written
    assert torch.equal(cache.k_cache[0, :, 3], k[0, :, 0])
    hip.device_error_word(DEV).zero_()


@pytest.mark.parametrize("rows,dim", [(1, 8192), (8, 8192), (64, 4096), (3, 2048), (16, 16384), (5, 264)])
@pytest.mark.parametrize("first_block", [False, True])
def test_ladder_norms_equals_two_add_rmsnorm_calls(hip, rows, dim, first_block):
    """lr_ladder_norms (both residual updates + both norms of a block in one launch) must give, bit for bit, what
    two lr_add_rmsnorm calls give, and match the oracle's block prologue (gpt_ladder_TP.py:326-354)."""
    x, d1, d2 = rnd(rows, dim, seed=50), rnd(rows, dim, seed=51, scale=0.3), rnd(rows, dim, seed=52, scale=0.3)
    g1, g2 = rnd(dim, seed=53), rnd(dim, seed=54)
    if first_block:
        d1 = d2 = None
    r_ref, n1_ref, n2_ref = torch.empty_like(x), torch.empty_like(x), torch.empty_like(x)
    hip.add_rmsnorm(x, d1, None, g1, r_ref, n1_ref, 1e-5)
    hip.add_rmsnorm(r_ref, d2, None, g2, r_ref, n2_ref, 1e-5)
    r, n1, n2 = x.clone(), torch.empty_like(x), torch.empty_like(x)
    hip.ladder_norms(r, d1, d2, g1, g2, r, n1, n2, 1e-5)       # residual updated in place
    assert torch.equal(r, r_ref) and torch.equal(n1, n1_ref) and torch.equal(n2, n2_ref)
    r1 = x if first_block else x + d1
    r2 = r1 if first_block else r1 + d2
    assert torch.equal(r, r2)
    assert_close_ulp(n1, O.rms_norm(r1, g1, 1e-5), max_ulp=2, max_frac=0.05, what="ladder_norms n1")
    assert_close_ulp(n2, O.rms_norm(r2, g2, 1e-5), max_ulp=2, max_frac=0.05, what="ladder_norms n2")


@pytest.mark.parametrize("M,D,K1,K2", [(33, 264, 2056, 4096), (64, 8192, 1024, 3584), (128, 2048, 2048, 8192), (100, 4096, 520, 14336),
                                       (300, 4104, 4096, 4104), (40, 16384, 8192, 512), (777, 2048, 256, 8192)])
def test_ladder_norms_of_partial_sums(hip, M, D, K1, K2):
    """Products left as partial sums and added by the norms: the bits of products finished first."""
    x, g1, g2 = rnd(M, D, seed=55), rnd(D, seed=56), rnd(D, seed=57)
    sums = [torch.empty(hip.linear_scratch_bytes(M), dtype=torch.uint8, device=DEV) for _ in range(2)]
    whole, parts = [], []
    for i, K in enumerate((K1, K2)):
        xi, w = rnd(M, K, seed=58 + i), rnd(D, K, seed=60 + i, scale=K ** -0.5)
        whole.append(hip.linear(xi, w, torch.empty(M, D, dtype=BF, device=DEV), scratch=sums[i]).clone())
        plan = hip.linear_plan(M, D, K)
        sums[i].fill_(255)                                       # (NaN, where a sum is not written)
        parts.append(hip.linear_pieces(xi, w, torch.empty(M, D, dtype=BF, device=DEV), sums[i]))
        assert isinstance(parts[-1], hip.Pieces) == (plan.cut > 0 and plan.whole == 0)
    outs = []
    for d1, d2 in (whole, parts):
        r, n1, n2 = x.clone(), torch.empty_like(x), torch.empty_like(x)
        hip.ladder_norms(r, d1, d2, g1, g2, r, n1, n2, 1e-5)
        outs.append((r, n1, n2))
    assert any(isinstance(p, hip.Pieces) for p in parts)
    for got, want in zip(outs[1], outs[0]):
        assert torch.equal(got, want)


class BlockBuffers:
    """The activation buffers of a model's workspace that ladder_blocks uses."""

    def __init__(self, hip, B, S, D, I, Hq, Hkv, hd):
        e = lambda c: torch.full((B * S, c), float("nan"), dtype=BF, device=DEV)
        self.B, self.S = B, S
        self.x, self.xn, self.xn2, self.a, self.m, self.y, self.act, self.h = (e(c) for c in (D, D, D, D, D, Hq * hd, I, 2 * I))
        self.qkv = e((Hq + 2 * Hkv) * hd)
        n = hip.linear_scratch_bytes(B * S)
        self.sums, self.sums_mlp = (torch.empty(n, dtype=torch.uint8, device=DEV) if n else None for _ in range(2))


# (rows without memory for sums; both pairs of products in a grid, in tiles of 64, 128 and 256 rows; none; K no whole k-tiles; several
# sequences; a block of its own)
@pytest.mark.parametrize("B,S,D,I,Hq,Hkv,hd,layers", [
    (1, 5, 256, 512, 4, 2, 64, 3), (2, 17, 512, 1024, 4, 1, 128, 3), (1, 63, 2048, 8192, 32, 8, 64, 2), (1, 128, 2048, 8192, 32, 8, 64, 3),
    (1, 130, 4096, 14336, 32, 8, 128, 2), (3, 100, 1032, 1096, 4, 2, 64, 3), (2, 256, 2048, 8192, 32, 8, 64, 2), (1, 1100, 1024, 3584, 8, 1, 128, 2),
    (1, 128, 2048, 8192, 32, 8, 64, 1), (1, 65, 2048, 8192, 32, 8, 64, 2), (2, 49, 2048, 8192, 32, 8, 64, 2),
])
def test_ladder_blocks_of_a_prompt(hip, B, S, D, I, Hq, Hkv, hd, layers):
    """Blocks in one call each against the calls they are made of.  Where only the order of fp32 sums differs, a rounded
    intermediate moves by a step of bf16 (2^-8) at the most, and few do: a stream of such blocks stays within 2^-7 by norm."""
    rows, Smax = B * S, S + 8
    pos = torch.arange(S, dtype=torch.int32, device=DEV)
    t = torch.outer(torch.arange(Smax, device=DEV).float(), 10000.0 ** (-torch.arange(0, hd, 2, device=DEV).float() / hd))
    table = torch.stack([t.cos(), t.sin()], -1).to(BF).contiguous()
    nqkv = (Hq + 2 * Hkv) * hd
    weights = []
    for i in range(layers):
        w = lambda k, n, m: rnd(n, m, seed=200 + 10 * i + k, scale=m ** -0.5)
        weights.append((1 + rnd(D, seed=208 + 10 * i, scale=0.1), 1 + rnd(D, seed=209 + 10 * i, scale=0.1), w(0, nqkv, D), w(1, D, Hq * hd),
                        w(2, 2 * I, D), w(3, D, I)))
    results = []
    for native in (True, True, False):
        ws = BlockBuffers(hip, B, S, D, I, Hq, Hkv, hd)
        ws.x.copy_(rnd(rows, D, seed=199))
        caches = [tuple(torch.zeros(B, Hkv, Smax, hd, dtype=BF, device=DEV) for _ in range(2)) for _ in range(layers)]
        if native:
            hip.ladder_blocks([(*w, *c) for w, c in zip(weights, caches)], ws, table, pos, Hq, Hkv, hd, 1e-5)
        else:
            a = m = None
            for (g1, g2, wqkv, wo, w1, w2), (kc, vc) in zip(weights, caches):
                hip.ladder_norms(ws.x, a, m, g1, g2, ws.x, ws.xn, ws.xn2, 1e-5)
                hip.linear_rope_kv(ws.xn, wqkv, ws.qkv, table, pos, kc, vc, B, S, Hq, Hkv, hd)
                hip.attn_prefill(ws.qkv, kc, vc, pos, ws.y, B, S, Hq, Hkv, hd)
                hip.linear(ws.y, wo, ws.a)
                hip.linear_swiglu_out(ws.xn2, w1, ws.act, ws.h)
                hip.linear(ws.act, w2, ws.m)
                a, m = ws.a, ws.m
        results.append([ws.x, ws.a, ws.m, *(t for c in caches for t in c)])
    for again, got, want in zip(*results):
        assert torch.equal(again, got) and torch.isfinite(got).all()
        assert (got.double() - want.double()).norm() <= 2.0 ** -7 * want.double().norm()


# (no product cut: 256 bytes; other tiles and pieces than with all the memory there may be; as many)
@pytest.mark.parametrize("rows,D,I,Hq,Hkv,hd", [(40, 1024, 3584, 8, 1, 128), (448, 2048, 8192, 32, 8, 64), (128, 2048, 8192, 32, 8, 64), (600, 2048, 8192, 32, 8, 64)])
def test_ladder_blocks_with_the_memory_that_a_model_gives_them(hip, rows, D, I, Hq, Hkv, hd):
    """A model's memory for partial sums is sized for its products one by one: fewer pieces may fit than with the most there
    may be, and no more is touched.  Only the order of fp32 sums differs: within 2^-7 by norm."""
    pos, N = torch.arange(rows, dtype=torch.int32, device=DEV), (Hq + 2 * Hkv) * hd
    table = O.rope_table(rows, hd, 10000.0, BF).to(DEV)
    w = lambda k, n, m: rnd(n, m, seed=220 + k, scale=m ** -0.5)
    weights = (1 + rnd(D, seed=228, scale=0.1), 1 + rnd(D, seed=229, scale=0.1), w(0, N, D), w(1, D, Hq * hd), w(2, 2 * I, D), w(3, D, I))
    sized = hip.linear_sums_bytes([(rows, N, D, False), (rows, D, Hq * hd, False), (rows, 2 * I, D, True), (rows, D, I, False)])
    results = []
    for nbytes in (hip.linear_scratch_bytes(rows), sized):
        ws = BlockBuffers(hip, 1, rows, D, I, Hq, Hkv, hd)
        held = [torch.full((nbytes + 4096,), 85, dtype=torch.uint8, device=DEV) for _ in range(2)]
        ws.sums, ws.sums_mlp = (h[:nbytes] for h in held)
        ws.x.copy_(rnd(rows, D, seed=219))
        caches = [[torch.zeros(1, Hkv, rows, hd, dtype=BF, device=DEV) for _ in range(2)] for _ in range(3)]
        hip.ladder_blocks([(*weights, *c) for c in caches], ws, table, pos, Hq, Hkv, hd, 1e-5)
        assert all((h[nbytes:] == 85).all() for h in held)
        results.append([ws.x, ws.a, ws.m, *(t for c in caches for t in c)])
    for got, want in zip(*results):
        assert torch.isfinite(got).all() and (got.double() - want.double()).norm() <= 2.0 ** -7 * want.double().norm()


@pytest.mark.parametrize("rows,dim,K", [(33, 1024, 8192), (64, 4096, 14336), (65, 2048, 8192), (130, 4096, 4096), (777, 4096, 14336), (48, 8192, 3584)])
@pytest.mark.parametrize("more", [False, True])
def test_add_rmsnorm_of_partial_sums(hip, rows, dim, K, more):
    """The bits of the product with its sum, then the norm."""
    x, w, gain = rnd(rows, K, seed=240), rnd(dim, K, seed=241, scale=K ** -0.5), 1 + rnd(dim, seed=242, scale=0.1)
    resid, d2 = rnd(rows, dim, seed=243), rnd(rows, dim, seed=244) if more else None
    sums = torch.empty(hip.linear_scratch_bytes(rows), dtype=torch.uint8, device=DEV)
    results = []
    for leave in (True, False):
        out = torch.empty(rows, dim, dtype=BF, device=DEV)
        d1 = (hip.linear_pieces if leave else hip.linear)(x, w, out, scratch=sums)
        assert isinstance(d1, hip.Pieces) == leave
        r, n = torch.empty_like(resid), torch.empty_like(resid)
        hip.add_rmsnorm(resid, d1, d2, gain, r, n, 1e-5)
        results.append((r, n))
    for got, want in zip(*results):
        assert torch.equal(got, want)


@pytest.mark.parametrize("M", [1, 2, 7, 8])
@pytest.mark.parametrize("N,K", [(5, 16), (1280, 4112), (2048, 528), (2056, 144), (4104, 2064)])
def test_bands_of_few_rows_equal_the_bands_of_many(hip, M, N, K):
    """Up to 8 input rows share fragments and thin bands load half a unit; a sum keeps its order, so a row's results are
    the bits it has in a call of 16 rows (inputs in whole lines, or e4m3 with full fragments)."""
    x = torch.full((16, K + 24), float("nan"), dtype=BF, device=DEV)[:, :K]      # rows and columns beyond are not read
    x.copy_(rnd(16, K, seed=90))
    w, w8 = rnd(N, K, seed=91), rnd(N, K, seed=92).to(torch.float8_e4m3fn)
    scales = rnd(N, seed=93).abs()
    few, many = (torch.empty(m, N, dtype=BF, device=DEV) for m in (M, 16))
    hip.linear_multi((x[:M], w, few, hip.EPI_NONE))
    hip.linear_multi((x, w, many, hip.EPI_NONE))
    assert torch.equal(few, many[:M])
    assert_close_ulp(few, linear_ref(x[:M], w), what="few rows")
    if M > 1:      # (one row of e4m3 weights is the matrix-vector kernel)
        hip.linear_fp8_multi((x[:M], w8, scales, few, hip.EPI_NONE))
        hip.linear_fp8_multi((x, w8, scales, many, hip.EPI_NONE))
        assert torch.equal(few, many[:M])


@pytest.mark.parametrize("M", [3, 24, 60])
@pytest.mark.parametrize("K", [8, 120, 136, 520, 8064, 8072, 8192, 8200, 16384, 16512])
def test_bands_in_slices_of_k(hip, M, K):
    """Each wave's slice of K: fewer chunks than waves, a last wave with fewer or none, slices of whole 4 KiB (which wrap around)."""
    x, w = rnd(M, K, seed=94), rnd(40, K, seed=95, scale=0.02)
    y = torch.empty(M, 40, dtype=BF, device=DEV)
    hip.linear_multi((x, w, y, hip.EPI_NONE))
    assert_close_ulp(y, linear_ref(x, w), what=f"slices M={M} K={K}")


@pytest.mark.parametrize("M", [3, 24, 60])
@pytest.mark.parametrize("K", [1024, 1032, 1536, 2048, 2056, 3072, 3080, 5120, 6144, 10240, 11008, 12280, 12296, 13312, 18432, 22016, 24576])
def test_bands_in_slices_of_k_and_in_turn(hip, M, K):
    """Widths on both sides of each line between the two; slices of whole 4 KiB (24576), which wrap around."""
    test_bands_in_slices_of_k(hip, M, K)


@pytest.mark.parametrize("M,N,K", [(33, 200, 64), (64, 136, 128), (40, 1030, 192), (64, 2000, 832), (48, 264, 8192), (64, 4096, 4160),
                                   (65, 200, 4096), (96, 264, 8192), (128, 1030, 8192), (127, 4104, 2112), (129, 200, 4160)])
@pytest.mark.parametrize("memory", [0, 8 << 20])
def test_products_in_long_rings(hip, M, N, K, memory):
    """Rings of three k-tiles: fewer k-tiles than slots, odd numbers of them, every column tile's own first k-tile, cut along K or not,
    rows on both sides of where they are used; columns beyond the last stay."""
    x, w = rnd(M, K, seed=96), rnd(N, K, seed=97, scale=0.02)
    scratch = torch.full((memory or 256,), 85, dtype=torch.uint8, device=DEV)
    y = torch.full((M, N + 8), 3.0, dtype=BF, device=DEV)
    hip.linear(x, w, y[:, :N], scratch=scratch)
    assert_close_ulp(y[:, :N].contiguous(), linear_ref(x, w), what=f"long ring M={M} N={N} K={K}")
    assert bool((y[:, N:] == 3.0).all())


@pytest.mark.parametrize("memory", [0, 8 << 20])
def test_products_in_long_rings_of_many_column_tiles(hip, memory):
    """More column tiles than k-tiles: several of them begin at the same one."""
    test_products_in_long_rings(hip, 48, 8200, 6656, memory)


@pytest.mark.parametrize("rows,dim", [(2, 4096), (2, 4104), (257, 8192), (3, 8200), (1, 16376)])
def test_norms_at_the_edges_of_the_lanes_per_row(hip, rows, dim):
    """256 lanes up to 4096 columns, 1024 above; the last columns leave most lanes of the last turn idle."""
    test_add_rmsnorm(hip, rows, dim)
    test_ladder_norms_equals_two_add_rmsnorm_calls(hip, rows, dim, False)


# ------------------------------------------------------------------------------------ weight-only fp8 linear

class Fp8Linear:
    def __init__(self, N, K, seed):
        self.weight, self.scales = rnd(N, K, seed=seed, scale=20.0).to(torch.float8_e4m3fn), rnd(N, seed=seed + 1).abs() * 1e-3

    def of(self, x):
        return (x.double() @ self.weight.double().T) * self.scales.double()


@pytest.mark.parametrize("M,N,K", [(17, 130, 128), (33, 264, 256), (64, 1030, 384), (40, 128, 640), (64, 1280, 8192), (20, 2048, 4096)])
@pytest.mark.parametrize("memory", [0, 8 << 20])
def test_linear_fp8_product(hip, M, N, K, memory):
    """17 to 64 rows of e4m3 weights in tiles: fewer k-tiles than the ring holds, odd numbers of them, ragged columns, cut along K or not."""
    x, lin = rnd(M, K, seed=110), Fp8Linear(N, K, 111)
    y = torch.full((M, N + 8), 3.0, dtype=BF, device=DEV)
    sums = torch.full((memory or 256,), 255, dtype=torch.uint8, device=DEV)
    assert hip.linear_fp8_product(x, lin, y[:, :N], sums)
    assert_close_ulp(y[:, :N].contiguous(), lin.of(x).to(BF), what=f"e4m3 product M={M} N={N} K={K}")
    assert bool((y[:, N:] == 3.0).all())


def test_linear_fp8_product_serves_17_to_64_rows_of_whole_k_tiles(hip):
    for M, K in ((16, 256), (65, 256), (32, 192)):
        assert not hip.linear_fp8_product(rnd(M, K), Fp8Linear(64, K, 1), torch.empty(M, 64, dtype=BF, device=DEV), None)


@pytest.mark.parametrize("B,Hq,Hkv,hd,D,memory", [(17, 8, 1, 128, 512, 8 << 20), (64, 4, 2, 64, 4096, 8 << 20), (33, 8, 2, 128, 256, 0)])
def test_linear_fp8_product_rotates_and_caches(hip, B, Hq, Hkv, hd, D, memory):
    """What the plain product followed by lr_rope_kv_write leaves, and no other cache slot touched."""
    Smax, block, pos_value = 48, 64, 37
    N = (Hq + 2 * Hkv) * hd
    x, lin, table = rnd(B, D, seed=40), Fp8Linear(N, D, 41), O.rope_table(block, hd, 10000.0, BF).to(DEV)
    pos = torch.tensor([pos_value], dtype=torch.int32, device=DEV)
    kc, vc = ([rnd(B, Hkv, Smax, hd, seed=s) for _ in range(2)] for s in (42, 43))
    q = torch.empty(2, B, N, dtype=BF, device=DEV)
    sums = torch.empty(memory or 256, dtype=torch.uint8, device=DEV)
    assert hip.linear_fp8_product(x, lin, q[0], sums)
    hip.rope_kv_write(q[0], table, False, pos, kc[0], vc[0], B, 1, Hq, Hkv, hd)
    assert hip.linear_fp8_product(x, lin, q[1], sums, hip.rope_kv_epilogue(table, pos, kc[1], vc[1], Hq, Hkv, hd))
    assert torch.equal(q[0], q[1]) and torch.equal(kc[0], kc[1]) and torch.equal(vc[0], vc[1])


@pytest.mark.parametrize("B,K,I", [(17, 128, 8192), (64, 8192, 456), (40, 4096, 1000)])
def test_attn_decode_beside_an_fp8_product(hip, B, K, I):
    """lr_attn_decode's bits, and the activation of the float64 product (up, gate and silu(gate) are each rounded: one step of any of them
    is at most 2^-7 of the result)."""
    Hq, Hkv, hd, Smax, pos = 8, 1, 128, 600, 555
    q, x, lin = rnd(B, (Hq + 2 * Hkv) * hd, seed=50), rnd(B, K, seed=53), Fp8Linear(2 * I, K, 54)
    kc, vc = rnd(B, Hkv, Smax, hd, seed=60), rnd(B, Hkv, Smax, hd, seed=80)
    p, tickets = torch.tensor([pos], dtype=torch.int32, device=DEV), torch.zeros(32 * B * Hq, dtype=torch.int32, device=DEV)
    scratch = torch.empty(hip.attn_decode_scratch_bytes(B, Hq, hd, Smax) // 4, dtype=torch.float32, device=DEV)
    y, act = torch.zeros(2, B, Hq * hd, dtype=BF, device=DEV), torch.empty(B, I, dtype=BF, device=DEV)
    hip.attn_decode(q, kc, vc, p, y[0], scratch, B, Hq, Hkv, hd)
    sums = torch.empty(max(hip.linear_fp8_product_bytes(B, 2 * I, K, True), 256), dtype=torch.uint8, device=DEV)
    assert hip.attn_decode_beside_product_fp8(q, kc, vc, p, y[1], scratch, B, Hq, Hkv, hd, tickets, x, lin, act, sums)
    assert torch.equal(y[0], y[1])
    u, g = lin.of(x).to(BF).float().chunk(2, 1)
    want = ((g / (1 + torch.exp(-g))).to(BF).float() * u).to(BF).float()
    assert ((act.float() - want).abs() <= 2.0 ** -7 * want.abs() + 1e-6 * want.abs().max()).all()


@pytest.mark.parametrize("M,D,K0,K1", [(17, 256, 128, 384), (64, 8192, 1024, 3584), (33, 4096, 4096, 14336)])
def test_fp8_pieces_of_two_products(hip, M, D, K0, K1):
    """Their sums, added in fp32, against the float64 products."""
    x, lins = [rnd(M, K, seed=120 + K) for K in (K0, K1)], [Fp8Linear(D, K, 130 + K) for K in (K0, K1)]
    n = hip.linear_fp8_pieces_two_bytes(M, D, K0, K1)
    sums = [torch.full((n,), 255, dtype=torch.uint8, device=DEV) for _ in range(2)]
    for x_, lin, p in zip(x, lins, hip.linear_fp8_pieces_two(x[0], lins[0], sums[0], x[1], lins[1], sums[1])):
        got = p.sums.view(torch.float32)[:p.count * M * D].view(p.count, M, D).double().sum(0)
        want = lin.of(x_)
        assert (got - want).abs().max() <= 2e-6 * want.abs().max() * x_.shape[1] ** 0.5


def test_linear_fp8_decodes_every_e4m3_value_exactly(hip):
    """All 254 finite byte patterns of float8_e4m3fn (normals, denormals, both zeros) through the kernel's
    conversion: with one-hot inputs and unit scales the output IS the stored value."""
    codes = torch.arange(256, dtype=torch.uint8, device=DEV)
    codes[0x7F] = 0          # the two NaN patterns are replaced
    codes[0xFF] = 0x80
    w8 = codes.view(torch.float8_e4m3fn).view(16, 16).contiguous()
    scales = torch.ones(16, dtype=BF, device=DEV)
    want = w8.to(torch.float32).T.contiguous()      # y[m, n] = w8[n, m]
    for m0 in (0, 8):
        x = torch.eye(16, dtype=BF, device=DEV)[m0:m0 + 8].contiguous()
        y = torch.empty(8, 16, dtype=BF, device=DEV)
        hip.linear_fp8(x, w8, scales, y)
        assert torch.equal(y.float(), want[m0:m0 + 8])
    assert want.abs().max().item() == 448.0 and (want.abs()[want != 0].min().item() == 2.0 ** -9)


@pytest.mark.parametrize("N,K", [(1280, 8192), (8192, 1024), (7168, 8192), (8192, 3584), (16032, 8192), (3072, 2048),
                                 (1001, 528), (24, 64)])
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 8, 16, 17, 300])
def test_linear_fp8(hip, M, N, K):
    """Decode (one row: matrix-vector kernel; 2 to 16 rows: matrix-core bands; fp8 weights streamed once; 17 rows: two passes
    of them, or as a prompt) and prefill (expanded to bf16 in scratch + matrix-core GEMM + column scaling) against the
    oracle's F.linear(x, w8.to(bf16)) * scales."""
    if M == 300 and N * K > 30e6:
        M = 65
    x = rnd(M, K, seed=40)
    w8, scales = O.quantize_fp8_rowwise(rnd(N, K, seed=41, scale=0.02, dtype=torch.float32), BF)
    y = torch.empty(M, N, dtype=BF, device=DEV)
    hip.linear_fp8(x, w8, scales, y)
    want = O.linear_fp8(x, w8, scales)
    # two roundings (the sum, then the scaled sum): a one-step difference in the first can survive as one or,
    # through double rounding, two steps of the result
    assert_close_ulp(y, want, max_ulp=2, max_frac=0.06, what=f"fp8 linear M={M} N={N} K={K}")
    exact = ((x.double() @ w8.double().T) * scales.double()).to(BF)
    # (the single rounding of the exact product differs from the two roundings of the scheme at about a quarter of the elements, by one step)
    assert_close_ulp(y, exact, max_ulp=2, max_frac=0.4, what="fp8 linear vs fp64")


@pytest.mark.parametrize("N,K,passes_to", [
    (2048, 1024, 32), (2040, 1040, 16), (2048, 1008, 16),    # columns and weights from which two passes are taken
    (2048, 2048, 48), (4096, 1008, 32),                      # and three
    (6144, 2736, 64), (6136, 2752, 48), (6144, 2720, 48),    # and four
    (7168, 8192, 64)])
@pytest.mark.parametrize("M", [17, 32, 33, 48, 49, 64, 65])
def test_linear_fp8_of_17_to_64_rows(hip, M, N, K, passes_to):
    """In passes of equal parts through the bands, the bits of linear_fp8_multi, or expanded, those of linear and the scaling; either
    against float64 (two roundings, as in test_linear_fp8)."""
    x = rnd(M, K, seed=40)
    w8, sc = O.quantize_fp8_rowwise(rnd(N, K, seed=41, scale=0.02, dtype=torch.float32), BF)
    y, want = torch.full((M, N + 8), 3.0, dtype=BF, device=DEV), torch.empty(M, N, dtype=BF, device=DEV)
    hip.linear_fp8(x, w8, sc, y[:, :N])
    if M <= passes_to:
        n, at = -(-M // 16), 0
        for left in range(n, 0, -1):
            rows = -(-(M - at) // left)
            hip.linear_fp8_multi((x[at:at + rows], w8, sc, want[at:at + rows], hip.EPI_NONE))
            at += rows
    else:
        hip.linear(x, w8.to(BF), want)
        want = (want.float() * sc.float()).to(BF)
    assert torch.equal(y[:, :N], want) and bool((y[:, N:] == 3.0).all())
    exact = ((x.double() @ w8.double().T) * sc.double()).to(BF)
    assert_close_ulp(y[:, :N].contiguous(), exact, max_ulp=2, max_frac=0.4, what="fp8 linear vs fp64")
    odd = torch.empty(M, N + 1, dtype=BF, device=DEV)     # rows that begin anywhere: expanded
    hip.linear_fp8(x, w8, sc, odd[:, :N])
    assert_close_ulp(odd[:, :N].contiguous(), exact, max_ulp=2, max_frac=0.4, what="fp8 linear vs fp64")


def test_linear_fp8_in_graphs_captured_one_after_the_other(hip):
    """A later graph's larger matrix, and memory given back in between, leave the earlier graphs' expanded weights where they were."""
    M = 80
    x = {K: rnd(M, K, seed=42) for K in (64, 2048)}
    cases = [O.quantize_fp8_rowwise(rnd(N, K, seed=43, scale=0.02, dtype=torch.float32), BF) for N, K in ((64, 64), (256, 2048), (4096, 2048))]
    want = [torch.empty(M, w8.shape[0], dtype=BF, device=DEV) for w8, _ in cases]
    eager = lambda: [hip.linear_fp8(x[w8.shape[1]], w8, sc, y) for (w8, sc), y in zip(cases, want)]
    eager()
    graphs = []
    for upto in (1, 2, 3):
        ys = [torch.zeros(M, w8.shape[0], dtype=BF, device=DEV) for w8, _ in cases[:upto]]
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            for (w8, sc), y in zip(cases, ys):
                hip.linear_fp8(x[w8.shape[1]], w8, sc, y)
        graphs.append((g, ys))
        torch.cuda.empty_cache()
    for _ in range(3):
        eager()
        for g, ys in graphs:
            for y in ys:
                y.fill_(3.0)
            g.replay()
            assert all(torch.equal(y, w) for y, w in zip(ys, want))


@pytest.mark.parametrize("M,D,Hq,Hkv,hd,I", [(1, 8192, 8, 1, 128, 3584), (8, 8192, 8, 1, 128, 3584), (3, 4096, 32, 8, 128, 1000),
                                             (5, 2048, 4, 2, 64, 72), (2, 1040, 2, 2, 64, 17), (4, 64, 1, 1, 8, 8),
                                             (16, 4096, 32, 8, 128, 14336), (13, 528, 4, 4, 64, 33)])
def test_linear_fp8_multi_equals_the_separate_calls(hip, M, D, Hq, Hkv, hd, I):
    """Two e4m3 projections per launch with their epilogues: q/k/v rotated and cached as lr_linear_fp8 followed by
    lr_rope_kv_write leaves them, up/gate as lr_linear_fp8 followed by lr_swiglu, plain projections as lr_linear_fp8
    -- bit for bit; rows (2p, 2p + 1) and (p, p + I) of one wave, K below and above the K-split thresholds."""
    Smax, block, pos_value = 40, 64, 23
    NQ = (Hq + 2 * Hkv) * hd
    xa, xb = rnd(M, D, seed=60), rnd(M, D, seed=61)
    wq, sq = O.quantize_fp8_rowwise(rnd(NQ, D, seed=62, scale=0.03, dtype=torch.float32), BF)
    w1, s1 = O.quantize_fp8_rowwise(rnd(2 * I, D, seed=63, scale=0.03, dtype=torch.float32), BF)
    table = O.rope_table(block, hd, 10000.0, BF).to(DEV)
    pos = torch.tensor([pos_value], dtype=torch.int32, device=DEV)
    kc = [rnd(M, Hkv, Smax, hd, seed=64) for _ in range(2)]
    vc = [rnd(M, Hkv, Smax, hd, seed=65) for _ in range(2)]
    # separate calls
    q_ref = torch.empty(M, NQ, dtype=BF, device=DEV)
    hip.linear_fp8(xa, wq, sq, q_ref)
    kv_proj = q_ref[:, Hq * hd:].clone()
    hip.rope_kv_write(q_ref, table, False, pos, kc[0], vc[0], M, 1, Hq, Hkv, hd)
    h = torch.empty(M, 2 * I, dtype=BF, device=DEV)
    hip.linear_fp8(xb, w1, s1, h)
    act_ref = F.silu(h[:, I:]) * h[:, :I]
    # one launch
    q = torch.empty(M, NQ, dtype=BF, device=DEV)
    act = torch.full((M, I), 3.0, dtype=BF, device=DEV)
    hip.linear_fp8_multi((xa, wq, sq, q, hip.rope_kv_epilogue(table, pos, kc[1], vc[1], Hq, Hkv, hd)),
                         (xb, w1, s1, act, hip.EPI_SWIGLU))
    if M == 1:   # the matrix-vector kernel: lr_linear_fp8's own sums
        assert torch.equal(q[:, :Hq * hd], q_ref[:, :Hq * hd]) and torch.equal(q[:, Hq * hd:], kv_proj)
        assert torch.equal(kc[1], kc[0]) and torch.equal(vc[1], vc[0])
        assert torch.equal(act, act_ref)
    else:        # from 2 rows on the matrix-core bands: another summation order, the same roundings
        assert_close_ulp(q, q_ref, max_ulp=2, max_frac=0.1, what="fp8 multi: q/k/v")
        keep = torch.ones(Smax, dtype=torch.bool, device=DEV)
        keep[pos_value] = False
        assert torch.equal(kc[1][:, :, keep], kc[0][:, :, keep]) and torch.equal(vc[1][:, :, keep], vc[0][:, :, keep])
        assert_close_ulp(kc[1][:, :, pos_value].contiguous(), kc[0][:, :, pos_value].contiguous(), max_ulp=2, max_frac=0.1,
                         what="fp8 multi: cached k")
        assert_close_ulp(vc[1][:, :, pos_value].contiguous(), vc[0][:, :, pos_value].contiguous(), max_ulp=2, max_frac=0.1,
                         what="fp8 multi: cached v")
        err = (act.float() - act_ref.float()).abs().max().item()
        assert err <= 2.0 ** -6 * act_ref.float().abs().max().item(), err
        assert (ulp_diff(act, act_ref) > 1).float().mean().item() < 0.05
    # plain projections, one of them with an odd number of rows
    wo, so = O.quantize_fp8_rowwise(rnd(D + 1, Hq * hd, seed=66, scale=0.03, dtype=torch.float32), BF) if (Hq * hd) % 16 == 0 \
        else (None, None)
    if wo is not None:
        y = rnd(M, Hq * hd, seed=67)
        a_ref, a = torch.empty(M, D + 1, dtype=BF, device=DEV), torch.zeros(M, D + 9, dtype=BF, device=DEV)
        hip.linear_fp8(y, wo, so, a_ref)
        m_ref, m = torch.empty(M, NQ, dtype=BF, device=DEV), torch.empty(M, NQ, dtype=BF, device=DEV)
        hip.linear_fp8(xa, wq, sq, m_ref)
        hip.linear_fp8_multi((y, wo, so, a[:, :D + 1], hip.EPI_NONE), (xa, wq, sq, m, hip.EPI_NONE))
        assert bool((a[:, D + 1:] == 0).all())
        if M == 1:
            assert torch.equal(a[:, :D + 1], a_ref) and torch.equal(m, m_ref)
        else:
            assert_close_ulp(a[:, :D + 1].contiguous(), a_ref, max_ulp=2, max_frac=0.1, what="fp8 multi: wo")
            assert_close_ulp(m, m_ref, max_ulp=2, max_frac=0.1, what="fp8 multi: second projection")


def test_rope_kv_write_position_out_of_range_sets_the_error_word(hip):
    """Positions beyond the cache or the RoPE table: the row is left alone, nothing lands in the cache and the
    per-device error word becomes LR_DEV_POS_RANGE (the reference raises an index error, utils.py:55)."""
    B, S, Smax, block, Hq, Hkv, hd = 1, 3, 16, 12, 2, 1, 64
    qkv = rnd(B, S, (Hq + 2 * Hkv) * hd, seed=29)
    before = qkv.clone()
    table = O.rope_table(block, hd, 10000, BF).to(DEV)
    kc = torch.zeros(B, Hkv, Smax, hd, dtype=BF, device=DEV)
    vc = torch.zeros_like(kc)
    word = hip.device_error_word(DEV)
    word.zero_()
    pos = torch.tensor([2, 16, 13], dtype=torch.int32, device=DEV)   # in range; beyond the cache; beyond the table
    hip.rope_kv_write(qkv, table, False, pos, kc, vc, B, S, Hq, Hkv, hd)
    torch.cuda.synchronize()
    assert word.item() == hip.DEV_POS_RANGE
    assert torch.equal(qkv[:, 1:], before[:, 1:]) and not torch.equal(qkv[:, 0], before[:, 0])
    assert bool((kc[:, :, 3:] == 0).all()) and bool((kc[:, :, 2] != 0).any())
    with pytest.raises(hip.LadderHipError):
        hip.raise_on_device_error(DEV)
    assert word.item() == 0      # reported once
    hip.raise_on_device_error(DEV)


# ------------------------------------------------------------------------------------ attention

@pytest.mark.parametrize("B,Hq,Hkv,hd,Smax,pos", [
    (1, 8, 1, 128, 2176, 2048), (1, 8, 1, 128, 2176, 0), (1, 8, 1, 128, 2176, 2175), (8, 8, 1, 128, 2176, 2100),
    (64, 8, 1, 128, 2176, 2111), (2, 32, 8, 128, 1280, 1033), (1, 32, 8, 64, 160, 131), (16, 16, 1, 128, 4160, 4100),
    (3, 4, 4, 64, 40, 17), (2, 8, 4, 128, 264, 200), (1, 16, 1, 128, 520, 519),
    # a cache long enough for more than 64 key chunks (merged by the general loop, not in one round trip), and
    # exactly 32 chunks
    (1, 8, 1, 128, 20000, 19000), (16, 8, 1, 128, 2048, 2047),
])
def test_attn_decode(hip, B, Hq, Hkv, hd, Smax, pos):
    q = rnd(B, Hq * hd, seed=21)
    kc = rnd(B, Hkv, Smax, hd, seed=22)
    vc = rnd(B, Hkv, Smax, hd, seed=23)
    kc[:, :, pos + 1:] = 7.0   # garbage beyond pos must not be read
    vc[:, :, pos + 1:] = -9.0
    p = torch.tensor([pos], dtype=torch.int32, device=DEV)
    y = torch.empty(B, Hq * hd, dtype=BF, device=DEV)
    scratch = torch.empty(hip.attn_decode_scratch_bytes(B, Hq, hd, Smax) // 4, dtype=torch.float32, device=DEV)
    hip.attn_decode(q, kc, vc, p, y, scratch, B, Hq, Hkv, hd)
    mask = (torch.arange(Smax, device=DEV) <= pos).view(1, Smax)
    want = O.sdpa_math(q.view(B, 1, Hq, hd).transpose(1, 2), kc, vc, mask).transpose(1, 2).reshape(B, Hq * hd)
    assert_close_ulp(y, want, max_frac=0.03, what="attn_decode")


@pytest.mark.parametrize("hd,Hq,Smax", [(128, 8, 64), (128, 16, 128), (64, 4, 129), (128, 2, 256), (64, 1, 2176)])
@pytest.mark.parametrize("pos", [0, 14, 15, 16, 63, 64, 65, 128, 200, 2175])
def test_attn_decode_chunk_edges_and_infinite_values(hip, hd, Hq, Smax, pos):
    """Positions at the edges of the 16-key tiles and 64-key groups, in chunks of two and of four groups; an infinite value comes
    through as the sum of positive weights times it, and stays in its dimension."""
    B, Hkv, pos = 3, 1, min(pos, Smax - 1)
    q, kc, vc = rnd(B, Hq * hd, seed=24), rnd(B, Hkv, Smax, hd, seed=25), rnd(B, Hkv, Smax, hd, seed=26)
    kc[:, :, pos + 1:] = 7.0
    vc[:, :, pos + 1:] = float("nan")
    p = torch.tensor([pos], dtype=torch.int32, device=DEV)
    scratch = torch.empty(hip.attn_decode_scratch_bytes(B, Hq, hd, Smax) // 4, dtype=torch.float32, device=DEV)
    mask = (torch.arange(Smax, device=DEV) <= pos).view(1, Smax)

    def want():
        v = vc.masked_fill(~mask.view(1, 1, Smax, 1), 0.0)
        return O.sdpa_math(q.view(B, 1, Hq, hd).transpose(1, 2), kc, v, mask).transpose(1, 2).reshape(B, Hq * hd)
    y = hip.attn_decode(q, kc, vc, p, torch.empty(B, Hq * hd, dtype=BF, device=DEV), scratch, B, Hq, Hkv, hd)
    assert_close_ulp(y, want(), max_frac=0.03, what="attn_decode")
    vc[1, 0, pos // 2, 5] = float("inf")
    vc[2, 0, pos, 9] = float("-inf")
    y, finite = hip.attn_decode(q, kc, vc, p, torch.empty_like(y), scratch, B, Hq, Hkv, hd), y
    y, finite = y.view(B, Hq, hd), finite.view(B, Hq, hd).clone()
    finite[1, :, 5], finite[2, :, 9] = float("inf"), float("-inf")
    assert torch.equal(y, finite)


@pytest.mark.parametrize("B,Hq,Hkv,hd,Smax,pos,D,I,epi_swiglu", [
    (8, 8, 1, 128, 2176, 2100, 1024, 456, True),     # the 70B rank shard's heads at batch 8
    (16, 32, 8, 128, 1100, 1024, 512, 1000, True),   # Ladder-8B's heads at batch 16
    (5, 4, 2, 64, 300, 0, 264, 72, True),            # first position: one key per sequence
    (16, 8, 8, 64, 520, 519, 136, 4100, False),      # one q head per kv head, a plain projection beside it
    (16, 16, 1, 128, 4224, 4100, 512, 456, True),    # the 405B rank shard's heads: 16 q heads as two groups of 8
    (3, 32, 2, 128, 200, 150, 264, 64, True),
    (1, 2, 1, 128, 64, 63, 64, 16, True),
])
def test_attn_decode_beside_equals_the_two_calls(hip, B, Hq, Hkv, hd, Smax, pos, D, I, epi_swiglu):
    """Attention items and projection bands in one grid: same bits as lr_attn_decode, then lr_linear_multi."""
    q = rnd(B, (Hq + 2 * Hkv) * hd, seed=50)         # q is the head of the fused q/k/v row, as in a decode step
    kc, vc = rnd(B, Hkv, Smax, hd, seed=51), rnd(B, Hkv, Smax, hd, seed=52)
    kc[:, :, pos + 1:] = 7.0
    vc[:, :, pos + 1:] = -9.0
    p = torch.tensor([pos], dtype=torch.int32, device=DEV)
    x = rnd(B, D, seed=53)
    w = rnd(2 * I if epi_swiglu else I, D, seed=54, scale=0.05)
    epi = hip.EPI_SWIGLU if epi_swiglu else hip.EPI_NONE
    nscr = hip.attn_decode_scratch_bytes(B, Hq, hd, Smax) // 4
    y, out = [torch.zeros(B, Hq * hd, dtype=BF, device=DEV) for _ in range(2)], \
        [torch.zeros(B, I, dtype=BF, device=DEV) for _ in range(2)]
    scratch = [torch.zeros(nscr, dtype=torch.float32, device=DEV) for _ in range(2)]
    hip.attn_decode(q, kc, vc, p, y[0], scratch[0], B, Hq, Hkv, hd)
    hip.linear_multi((x, w, out[0], epi))
    assert hip.attn_decode_beside(q, kc, vc, p, y[1], scratch[1], B, Hq, Hkv, hd, (x, w, out[1], epi))
    assert torch.equal(y[1], y[0]) and torch.equal(out[1], out[0])
    mask = (torch.arange(Smax, device=DEV) <= pos).view(1, Smax)
    want = O.sdpa_math(q[:, :Hq * hd].reshape(B, 1, Hq, hd).transpose(1, 2), kc, vc, mask).transpose(1, 2)
    assert_close_ulp(y[1], want.reshape(B, Hq * hd), max_frac=0.03, what="attn_decode_beside")


@pytest.mark.parametrize("B,Hq,Hkv,hd,Smax,pos,D,I", [(8, 8, 1, 128, 2176, 2100, 8192, 456), (2, 8, 1, 128, 600, 599, 1024, 200),
                                                    (16, 32, 8, 128, 300, 17, 512, 72), (5, 16, 1, 128, 520, 400, 2048, 40),
                                                    (4, 4, 2, 64, 100, 99, 272, 24)])
def test_attn_decode_beside_fp8_equals_the_two_calls(hip, B, Hq, Hkv, hd, Smax, pos, D, I):
    """Attention items and the bands of an e4m3 up/gate projection in one grid: same bits as lr_attn_decode, then
    lr_linear_fp8_multi; a single row is declined."""
    q = rnd(B, (Hq + 2 * Hkv) * hd, seed=70)
    kc, vc = rnd(B, Hkv, Smax, hd, seed=71), rnd(B, Hkv, Smax, hd, seed=72)
    p = torch.tensor([pos], dtype=torch.int32, device=DEV)
    x = rnd(B, D, seed=73)
    w8, sc = O.quantize_fp8_rowwise(rnd(2 * I, D, seed=74, scale=0.05, dtype=torch.float32), BF)
    nscr = hip.attn_decode_scratch_bytes(B, Hq, hd, Smax) // 4
    y = [torch.zeros(B, Hq * hd, dtype=BF, device=DEV) for _ in range(2)]
    out = [torch.zeros(B, I, dtype=BF, device=DEV) for _ in range(2)]
    scratch = [torch.zeros(nscr, dtype=torch.float32, device=DEV) for _ in range(2)]
    hip.attn_decode(q, kc, vc, p, y[0], scratch[0], B, Hq, Hkv, hd)
    hip.linear_fp8_multi((x, w8, sc, out[0], hip.EPI_SWIGLU))
    assert hip.attn_decode_beside_fp8(q, kc, vc, p, y[1], scratch[1], B, Hq, Hkv, hd, (x, w8, sc, out[1], hip.EPI_SWIGLU))
    assert torch.equal(y[1], y[0]) and torch.equal(out[1], out[0])
    assert out[1].float().abs().sum().item() > 0
    o1 = torch.full((1, I), 5.0, dtype=BF, device=DEV)
    y1 = torch.full((1, Hq * hd), 5.0, dtype=BF, device=DEV)
    assert not hip.attn_decode_beside_fp8(q[:1], kc[:1], vc[:1], p, y1, scratch[1], 1, Hq, Hkv, hd,
                                          (x[:1], w8, sc, o1, hip.EPI_SWIGLU))
    torch.cuda.synchronize()
    assert bool((o1 == 5.0).all()) and bool((y1 == 5.0).all())


@pytest.mark.parametrize("looks", [0, 1, 3])   # the library's own number; a merging wave that does not wait at all; one that looks twice
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("B,Hq,Hkv,hd,Smax,pos", [
    (8, 8, 1, 128, 2176, 2100),      # 32 chunks, the whole first round trip
    (3, 4, 4, 64, 4096, 4095),       # more than 32 chunks: two round trips; one q head per kv head
    (2, 8, 1, 128, 4096, 40),        # 64 chunks, most of them without a key
    (16, 32, 8, 128, 1100, 1024),    # few chunks, several kv heads
    (5, 16, 1, 128, 520, 400),       # 16 q heads as two groups of 8
    (4, 8, 2, 64, 40, 0),            # one chunk, one key
    (2, 8, 1, 128, 20000, 19000),    # more chunks than the merge inside the launch takes: a launch of its own
])
def test_attn_decode_merged_beside_a_projection_equals_the_two_launches(hip, looks, fp8, B, Hq, Hkv, hd, Smax, pos):
    """The chunks merged by waves at the end of the grid, or, where these do not wait for them, by the item that stores a kv head's
    last one: the bits of the merge in a launch of its own, launch after launch, with scratch of NaN (nothing is read that this
    call has not written), and the tickets zero again."""
    D, I = 272, 72
    q = rnd(B, (Hq + 2 * Hkv) * hd, seed=50)
    p = torch.tensor([pos], dtype=torch.int32, device=DEV)
    x = rnd(B, D, seed=53)
    w = rnd(2 * I, D, seed=54, scale=0.05, dtype=torch.float32)
    if fp8:
        proj, beside, alone = (x, *O.quantize_fp8_rowwise(w, BF)), hip.attn_decode_beside_fp8, hip.linear_fp8_multi
    else:
        proj, beside, alone = (x, w.to(BF)), hip.attn_decode_beside, hip.linear_multi
    tickets = torch.zeros(B * Hq, 32, dtype=torch.int32, device=DEV)
    tickets[:, 1] = looks
    scratch = torch.empty(hip.attn_decode_scratch_bytes(B, Hq, hd, Smax) // 4, dtype=torch.float32, device=DEV)
    for seed in range(4):
        kc, vc = rnd(B, Hkv, Smax, hd, seed=60 + seed), rnd(B, Hkv, Smax, hd, seed=80 + seed)
        y, out = torch.zeros(2, B, Hq * hd, dtype=BF, device=DEV), torch.zeros(2, B, I, dtype=BF, device=DEV)
        hip.attn_decode(q, kc, vc, p, y[0], scratch, B, Hq, Hkv, hd)
        alone((*proj, out[0], hip.EPI_SWIGLU))
        scratch.fill_(float("nan"))
        assert beside(q, kc, vc, p, y[1], scratch, B, Hq, Hkv, hd, (*proj, out[1], hip.EPI_SWIGLU), tickets)
        assert torch.equal(y[1], y[0]) and torch.equal(out[1], out[0]) and bool(y[0].any())
        assert not bool(tickets[:, 0].any())
    assert looks != 1 or Smax == 20000 or bool(tickets[:, 2].any())   # (an item takes microseconds: some waves were earlier)


@pytest.mark.parametrize("looks", [0, 1, 3])
@pytest.mark.parametrize("B,Hq,Hkv,hd,Smax,pos,K,I", [
    (64, 8, 1, 128, 2176, 2100, 2048, 456),      # chunks of four groups of keys, a product in pieces
    (33, 8, 2, 64, 640, 300, 1024, 17),          # one row more than the bands', one pair of a tile's 64
    (64, 16, 1, 128, 128, 5, 64, 24000),         # 16 q heads as two groups of 8; whole tiles, more than the chip has CUs
    (40, 4, 4, 64, 200, 199, 4096, 1000),        # one q head per kv head
])
def test_attn_decode_beside_a_product_equals_the_two_calls(hip, looks, B, Hq, Hkv, hd, Smax, pos, K, I):
    """Tiles, attention items and their merge in one grid, with and without a wait for the items: the bits of lr_attn_decode and
    lr_linear_swiglu_out, launch after launch, the tickets zero again."""
    q, x = rnd(B, (Hq + 2 * Hkv) * hd, seed=50), rnd(B, K, seed=53)
    w = rnd(2 * I, K, seed=54, scale=K ** -0.5)
    p = torch.tensor([pos], dtype=torch.int32, device=DEV)
    tickets = torch.zeros(B * Hq, 32, dtype=torch.int32, device=DEV)
    tickets[:, 1] = looks
    scratch = torch.empty(hip.attn_decode_scratch_bytes(B, Hq, hd, Smax) // 4, dtype=torch.float32, device=DEV)
    sums = torch.empty(hip.linear_scratch_bytes(B), dtype=torch.uint8, device=DEV)
    for seed in range(3):
        kc, vc = rnd(B, Hkv, Smax, hd, seed=60 + seed), rnd(B, Hkv, Smax, hd, seed=80 + seed)
        y = torch.zeros(2, B, Hq * hd, dtype=BF, device=DEV)
        act = [torch.full((B, I + 3), 5.0, dtype=BF, device=DEV) for _ in range(2)]
        hip.attn_decode(q, kc, vc, p, y[0], scratch, B, Hq, Hkv, hd)
        hip.linear_swiglu_out(x, w, act[0][:, :I], sums=sums)
        scratch.fill_(float("nan"))
        sums.fill_(255)
        assert hip.attn_decode_beside_product(q, kc, vc, p, y[1], scratch, B, Hq, Hkv, hd, tickets, x, w, act[1][:, :I], sums)
        assert torch.equal(y[1], y[0]) and torch.equal(act[1], act[0]) and bool(y[0].any())
        assert not bool(tickets[:, 0].any())


@pytest.mark.parametrize("B,K,I", [(17, 64, 8192), (32, 8192, 456), (20, 4096, 1000)])
def test_attn_decode_beside_a_product_of_up_to_32_rows(hip, B, K, I):
    """Rows that lr_linear_swiglu_out gives the bands: lr_attn_decode's bits, and the activation of the float64 product (up, gate and
    silu(gate) are each rounded: one step of any of them is at most 2^-7 of the result)."""
    Hq, Hkv, hd, Smax, pos = 8, 1, 128, 600, 555
    q, x, w = rnd(B, (Hq + 2 * Hkv) * hd, seed=50), rnd(B, K, seed=53), rnd(2 * I, K, seed=54, scale=K ** -0.5)
    kc, vc = rnd(B, Hkv, Smax, hd, seed=60), rnd(B, Hkv, Smax, hd, seed=80)
    p, tickets = torch.tensor([pos], dtype=torch.int32, device=DEV), torch.zeros(32 * B * Hq, dtype=torch.int32, device=DEV)
    scratch = torch.empty(hip.attn_decode_scratch_bytes(B, Hq, hd, Smax) // 4, dtype=torch.float32, device=DEV)
    y, act = torch.zeros(2, B, Hq * hd, dtype=BF, device=DEV), torch.empty(B, I, dtype=BF, device=DEV)
    hip.attn_decode(q, kc, vc, p, y[0], scratch, B, Hq, Hkv, hd)
    sums = torch.empty(200 << 15, dtype=torch.uint8, device=DEV)
    assert hip.attn_decode_beside_product(q, kc, vc, p, y[1], scratch, B, Hq, Hkv, hd, tickets, x, w, act, sums)
    assert torch.equal(y[0], y[1])
    u, g = (x.double() @ w.double().T).to(BF).float().chunk(2, 1)
    want = ((g / (1 + torch.exp(-g))).to(BF).float() * u).to(BF).float()
    assert ((act.float() - want).abs() <= 2.0 ** -7 * 3 * want.abs() + 2.0 ** -12).all()


def test_attn_decode_beside_a_product_declines_what_it_has_no_kernel_for(hip):
    """Rows that the bands or larger tiles serve, K of no whole k-tiles, more key chunks than a wave merges: False, nothing launched."""
    def run(B, K=4096, Smax=64, Hq=8):
        hd, I = 64, 64
        kc, vc = rnd(B, 1, Smax, hd, seed=56), rnd(B, 1, Smax, hd, seed=57)
        y, act = torch.full((B, Hq * hd), 5.0, dtype=BF, device=DEV), torch.full((B, I), 5.0, dtype=BF, device=DEV)
        scratch = torch.zeros(hip.attn_decode_scratch_bytes(B, Hq, hd, Smax) // 4, dtype=torch.float32, device=DEV)
        ok = hip.attn_decode_beside_product(rnd(B, Hq * hd, seed=55), kc, vc, torch.tensor([3], dtype=torch.int32, device=DEV), y, scratch, B, Hq, 1,
                                            hd, torch.zeros(32 * B * Hq, dtype=torch.int32, device=DEV), rnd(B, K, seed=58), rnd(2 * I, K, seed=59),
                                            act, None)
        return ok, bool((y == 5.0).all()) and bool((act == 5.0).all())
    assert run(33)[0] is True
    for kw in (dict(B=16), dict(B=65), dict(B=33, K=4104), dict(B=33, Smax=17000), dict(B=33, Hq=3)):
        assert run(**kw) == (False, True), kw


@pytest.mark.parametrize("M,N,K0,K1,joint", [(64, 8192, 1024, 3584, True), (33, 264, 2048, 4096, True), (128, 2048, 2048, 8192, True),
                                             (64, 2048, 64, 64, True), (17, 8192, 1024, 3584, True), (32, 260, 4096, 64, True),
                                             (64, 16384, 2048, 6656, True),
                                             (16, 264, 2048, 4096, False), (33, 264, 2056, 4096, False)])   # (few rows; no whole k-tiles)
def test_linear_pieces_two(hip, monkeypatch, M, N, K0, K1, joint):
    """Two products' partial sums of one grid, or of two where the library declines: their totals, in fp32, against float64."""
    x, w = [rnd(M, K, seed=90 + K % 7) for K in (K0, K1)], [rnd(N, K, seed=91 + K % 7, scale=K ** -0.5) for K in (K0, K1)]
    n = hip.linear_pieces_two_bytes(M, N, K0, K1)
    assert (n > 0) == joint
    sums = [torch.full((max(hip.linear_scratch_bytes(M), n, 256),), 255, dtype=torch.uint8, device=DEV) for _ in range(2)]
    out = [torch.zeros(M, N, dtype=BF, device=DEV) for _ in range(2)]
    apart, single = [], hip.linear_pieces
    monkeypatch.setattr(hip, "linear_pieces", lambda *a: (apart.append(a), single(*a))[1])
    parts = hip.linear_pieces_two(x[0], w[0], out[0], sums[0], x[1], w[1], out[1], sums[1])
    assert len(apart) == (0 if joint else 2)
    for i, p in enumerate(parts):
        want = x[i].double() @ w[i].double().T
        assert not joint or isinstance(p, hip.Pieces) and p.count * M * N * 4 <= n and not bool(out[i].any())
        if isinstance(p, hip.Pieces):
            got = sums[i].view(torch.float32)[:p.count * M * N].view(p.count, M, N).double().sum(0)
            assert ((got - want).abs() <= 1e-5 * want.abs().max()).all()
        else:
            assert_close_ulp(p, want.to(BF))


def test_attn_decode_beside_declines_what_it_has_no_kernel_for(hip):
    """More than 16 rows, 32 q heads per kv head, or a projection that writes the cache: False, nothing launched."""
    def run(B, Hq, Hkv, epi=None):
        hd, Smax, D, I = 128, 64, 64, 16
        q = rnd(B, Hq * hd, seed=55)
        kc, vc = rnd(B, Hkv, Smax, hd, seed=56), rnd(B, Hkv, Smax, hd, seed=57)
        p = torch.tensor([3], dtype=torch.int32, device=DEV)
        y = torch.full((B, Hq * hd), 5.0, dtype=BF, device=DEV)
        N = (Hq + 2 * Hkv) * hd if epi is not None else I
        out = torch.full((B, N), 5.0, dtype=BF, device=DEV)
        scratch = torch.zeros(hip.attn_decode_scratch_bytes(B, Hq, hd, Smax) // 4, dtype=torch.float32, device=DEV)
        if epi is not None:
            epi = hip.rope_kv_epilogue(O.rope_table(64, hd, 10000.0, BF).to(DEV), p, kc, vc, Hq, Hkv, hd)
        ok = hip.attn_decode_beside(q, kc, vc, p, y, scratch, B, Hq, Hkv, hd,
                                    (rnd(B, D, seed=58), rnd(N, D, seed=59), out, hip.EPI_NONE if epi is None else epi))
        torch.cuda.synchronize()
        return ok, bool((y == 5.0).all()) and bool((out == 5.0).all())
    assert run(17, 8, 1) == (False, True)
    assert run(4, 32, 1) == (False, True)
    assert run(4, 8, 1, epi="rope") == (False, True)
    assert run(4, 8, 1)[0] is True


@pytest.mark.parametrize("B,S,Hq,Hkv,hd,Smax,start", [
    (1, 128, 8, 1, 128, 136, 0), (2, 100, 4, 2, 64, 160, 0), (1, 300, 8, 1, 128, 512, 100), (1, 2048, 8, 1, 128, 2176, 0),
    (3, 65, 32, 8, 64, 72, 0),
    # one q head per kv head (4 query tiles per workgroup), odd group sizes, 16 heads per kv head, S below the
    # matrix-core kernel's threshold, a single query tile with a long history
    (2, 130, 4, 4, 128, 136, 0), (1, 97, 6, 2, 64, 104, 3), (1, 64, 16, 1, 128, 64, 0), (2, 9, 8, 2, 64, 16, 0),
    (1, 17, 8, 1, 128, 1024, 1000),
])
def test_attn_prefill(hip, B, S, Hq, Hkv, hd, Smax, start):
    q = rnd(B, S, Hq * hd, seed=24)
    kc = rnd(B, Hkv, Smax, hd, seed=25)
    vc = rnd(B, Hkv, Smax, hd, seed=26)
    pos = torch.arange(start, start + S, dtype=torch.int32, device=DEV)
    y = torch.empty(B, S, Hq * hd, dtype=BF, device=DEV)
    hip.attn_prefill(q, kc, vc, pos, y, B, S, Hq, Hkv, hd)
    mask = torch.arange(Smax, device=DEV).view(1, Smax) <= pos.view(S, 1)
    want = O.sdpa_math(q.view(B, S, Hq, hd).transpose(1, 2), kc, vc, mask).transpose(1, 2).reshape(B, S, Hq * hd)
    assert_close_ulp(y, want, max_frac=0.03, what="attn_prefill")


# (portions of 32 and of 64 keys, with and without a last half, and each wave half of them; workgroups of one, two and four heads, in
# columns that are a multiple of eight and that are not)
@pytest.mark.parametrize("B,S,Hq,Hkv,hd,start", [
    (1, 16, 4, 1, 128, 0), (2, 33, 8, 2, 128, 31), (1, 128, 6, 3, 128, 64), (1, 129, 32, 8, 128, 0), (3, 161, 2, 2, 128, 95), (1, 511, 8, 2, 128, 1),
    (1, 512, 8, 1, 128, 0), (1, 545, 6, 3, 128, 63), (2, 600, 2, 2, 128, 200), (8, 520, 32, 8, 128, 0), (5, 610, 28, 7, 128, 17),
    (1, 17, 4, 1, 64, 0), (1, 130, 6, 3, 64, 33), (1, 512, 32, 8, 64, 0), (1, 577, 2, 2, 64, 64), (8, 530, 32, 8, 64, 3)])
def test_attn_prefill_portions_of_keys(hip, B, S, Hq, Hkv, hd, start):
    """Nothing beyond the last position is used, whatever lies there."""
    n = start + S
    q, kc, vc = rnd(B, S, Hq * hd, seed=31), rnd(B, Hkv, n + 70, hd, seed=32), rnd(B, Hkv, n + 70, hd, seed=33)
    kc[:, :, n:], vc[:, :, n:] = float("nan"), float("nan")
    pos = torch.arange(start, n, dtype=torch.int32, device=DEV)
    y = torch.full((B, S, Hq * hd), float("nan"), dtype=BF, device=DEV)
    hip.attn_prefill(q, kc, vc, pos, y, B, S, Hq, Hkv, hd)
    mask = torch.arange(n, device=DEV).view(1, n) <= pos.view(S, 1)
    want = O.sdpa_math(q.view(B, S, Hq, hd).transpose(1, 2), kc[:, :, :n].contiguous(), vc[:, :, :n].contiguous(), mask)
    assert_close_ulp(y, want.transpose(1, 2).reshape(B, S, Hq * hd), max_frac=0.03, what="attn_prefill, portions")


# (one key, 32 and 33 of them, alone and behind others, where they are computed as half a portion and where they are not)
@pytest.mark.parametrize("B,S,Hq,Hkv,hd,start", [
    (1, 16, 4, 1, 128, 17), (2, 32, 8, 2, 128, 0), (1, 32, 4, 1, 128, 64), (1, 65, 8, 2, 128, 0), (3, 97, 8, 8, 128, 0), (1, 96, 6, 3, 128, 0),
    (1, 33, 6, 3, 128, 64), (1, 97, 4, 2, 128, 63), (2, 32, 8, 2, 64, 0), (1, 33, 4, 1, 64, 0), (1, 65, 6, 3, 64, 0), (3, 96, 2, 2, 64, 0),
    (1, 128, 4, 1, 64, 1), (1, 129, 4, 1, 64, 0), (1, 129, 4, 4, 64, 31)])
def test_attn_prefill_last_portion_of_keys(hip, B, S, Hq, Hkv, hd, start):
    test_attn_prefill_portions_of_keys(hip, B, S, Hq, Hkv, hd, start)


@pytest.mark.parametrize("qscale", [4.0, 12.0])
def test_attn_prefill_large_scores(hip, qscale):
    """Scores with a standard deviation of 4 and 12: the running maximum of a query jumps by more than the kernel lets
    its reference point lag, on tiles late in the history too, so accumulators are rescaled in mid-stream; and the
    softmax is nearly one-hot at the larger scale."""
    B, S, Hq, Hkv, hd, Smax = 2, 700, 8, 2, 128, 704
    q = rnd(B, S, Hq * hd, seed=124, scale=qscale)
    kc = rnd(B, Hkv, Smax, hd, seed=125)
    vc = rnd(B, Hkv, Smax, hd, seed=126)
    pos = torch.arange(S, dtype=torch.int32, device=DEV)
    y = torch.empty(B, S, Hq * hd, dtype=BF, device=DEV)
    hip.attn_prefill(q, kc, vc, pos, y, B, S, Hq, Hkv, hd)
    mask = torch.arange(Smax, device=DEV).view(1, Smax) <= pos.view(S, 1)
    want = O.sdpa_math(q.view(B, S, Hq, hd).transpose(1, 2), kc, vc, mask).transpose(1, 2).reshape(B, S, Hq * hd)
    assert_close_ulp(y, want, max_frac=0.03, what="attn_prefill, large scores")


def test_attn_prefill_equal_sequences_give_equal_rows(hip):
    """Eight copies of one sequence: every copy's output is the same bit pattern, on repeated calls too (the kernel
    has no race and reads no register before its producer has finished)."""
    B, S, Hq, Hkv, hd, Smax = 8, 1024, 32, 8, 128, 1072
    q = rnd(1, S, Hq * hd, seed=224).repeat(B, 1, 1).contiguous()
    kc = rnd(1, Hkv, Smax, hd, seed=225).repeat(B, 1, 1, 1).contiguous()
    vc = rnd(1, Hkv, Smax, hd, seed=226).repeat(B, 1, 1, 1).contiguous()
    pos = torch.arange(S, dtype=torch.int32, device=DEV)
    first = None
    for _ in range(3):
        y = torch.empty(B, S, Hq * hd, dtype=BF, device=DEV)
        hip.attn_prefill(q, kc, vc, pos, y, B, S, Hq, Hkv, hd)
        assert all(torch.equal(y[0], y[b]) for b in range(1, B))
        first = y if first is None else first
        assert torch.equal(y, first)


# ------------------------------------------------------------------------------------ argmax

def test_argmax_lowest_index_on_ties(hip):
    B, V = 4, 128256
    lg = rnd(B, V, seed=27, scale=0.04)
    lg[0, [77, 100000]] = 5.0
    lg[1, [128255, 5]] = 5.0
    lg[2, 128255] = 9.0
    out = torch.empty(B, 1, dtype=torch.int32, device=DEV)
    hip.argmax(lg, out)
    want = torch.argmax(lg, dim=-1, keepdim=True).to(torch.int32)
    assert torch.equal(out, want) and out.flatten().tolist()[:3] == [77, 5, 128255]
    # last position of [B, S, V] logits: a strided [B, V] view; and a vocab that is not a multiple of 8
    lg3 = rnd(2, 3, 1008, seed=28)
    hip.argmax(lg3[:, -1, :1003], out[:2])
    assert torch.equal(out[:2], lg3[:, -1, :1003].argmax(-1, keepdim=True).to(torch.int32))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("V", [1, 7, 8, 9, 1003, 8191, 8192, 8200, 65536, 65543, 128256])
def test_argmax_at_the_edges_of_its_groups(hip, V, dtype):
    """Whole and partial groups of 8 and rounds of 8192 and 65536 columns; ties, signed zeros, infinities, NaNs (never
    chosen) and rows without a value above the lowest one."""
    g = torch.Generator().manual_seed(V)
    lg = (torch.randint(-40, 40, (9, V), generator=g) / 8).to(dtype)   # (many equal values)
    lg[1] = -0.0
    lg[1, V // 2:] = 0.0
    lg[2] = float("-inf")
    lg[3] = float("nan")
    lg[4, ::2] = float("nan")
    lg[5, V // 3:] = float("inf")
    lg[6] = float("-inf")
    lg[6, : V // 2] = float("nan")
    lg[7, V - 1] = 9.0
    lg[8, :] = -3.0e38
    want = torch.argmax(torch.where(lg.isnan(), float("-inf"), lg.double()), -1)
    want = torch.where(lg.isnan().all(-1), 0, want)
    want[6] = min(V // 2, V - 1)
    ld = (V + 15) // 8 * 8
    padded = torch.full((9, ld), 1e9, dtype=dtype, device=DEV)      # (columns beyond V are not the row's)
    padded[:, :V] = lg.to(DEV)
    out = torch.full((9, 1), -7, dtype=torch.int32, device=DEV)
    hip.argmax(padded[:, :V], out)
    assert out.flatten().tolist() == want.tolist()


def test_argmax_of_a_row_as_long_as_its_index_reaches(hip):
    """Columns whose steps pass 2^31: the last one, in the ragged end, the last of the groups of eight, one in the middle; none at all."""
    V = 2 ** 31 - 9
    lg, out = torch.full((1, V + 1), -1.0, dtype=BF, device=DEV), torch.empty(1, dtype=torch.int32, device=DEV)
    for at in (V - 1, V - 8, V // 2):
        lg[0, at] = 1.0
        hip.argmax(lg[:, :V], out)
        assert out.item() == at
        lg[0, at] = float("-inf")
    lg.fill_(float("-inf"))
    hip.argmax(lg[:, :V], out)
    assert out.item() == 0


def test_torch_argmax_itself_returns_first_maximum_on_this_device():
    """The oracle's greedy() relies on it."""
    lg = torch.zeros(1, 16032, dtype=BF, device=DEV)
    lg[0, [15000, 40, 9000]] = 1.0
    assert torch.argmax(lg, -1).item() == 40


# ------------------------------------------------------------------------------------ stream read

def test_stream_read_runs_and_leaves_the_sink_alone(hip):
    """The measurement aid reads the buffer and writes nothing (the xor of the data is not the magic value)."""
    buf = torch.full((64 << 20,), 3, dtype=torch.uint8, device=DEV)
    sink = torch.full((1,), 1234, dtype=torch.int32, device=DEV)
    for _ in range(3):
        hip.stream_read(buf, sink)
    torch.cuda.synchronize()
    assert sink.item() == 1234
    with pytest.raises(hip.LadderHipError):
        hip.stream_read(buf[:1024], sink)


# ------------------------------------------------------------------------------------ the prefill GEMM's tiles and pieces

@pytest.mark.parametrize("M,N,K", [
    (33, 264, 520), (64, 1280, 8192), (40, 24, 64),      # decode batches: with memory for sums 64-row tiles
    (65, 8, 8), (100, 72, 64), (129, 264, 520), (256, 256, 128), (257, 512, 192), (300, 520, 200), (513, 40, 4096),
    (777, 1032, 1000),                                   # 64-row tiles: a row, column or k too many; odd numbers of k-tiles
    (128, 1024, 8192), (300, 2048, 4160), (777, 2048, 7168),   # cut along K where there is memory for it: tiles of 64 x 128,
    (2100, 2560, 8192),                                        # 128 x 128, 128 x 256 and 256 x 256
])
def test_linear_tiles_and_pieces(hip, M, N, K):
    """Whole tiles, and tiles cut along K with their sums added by a second launch, against the float64 product: fp32
    accumulation and one rounding either way (the assert allows the rounding to fall on the other side).  The cut form
    repeats bit for bit and writes no row or column beyond its own."""
    x, w = rnd(M, K, seed=90), rnd(N, K, seed=91, scale=K ** -0.5)
    want = (x.double() @ w.double().T).to(BF)
    sums = torch.empty(hip.linear_scratch_bytes(M), dtype=torch.uint8, device=DEV)
    outs = []
    for scratch in (None, sums, sums):
        y = torch.full((M + 1, N + 8), 5.0, dtype=BF, device=DEV)
        hip.linear(x, w, y[:M, :N], scratch=scratch)
        assert_close_ulp(y[:M, :N].contiguous(), want, what=f"{M} x {N} x {K}")
        assert (y[M:] == 5.0).all() and (y[:, N:] == 5.0).all()
        outs.append(y)
    assert torch.equal(outs[1], outs[2])


def gemm_kind(plan):
    return (plan.tile_rows, plan.tile_cols), "whole" if not plan.cut else "mixed" if plan.whole else "cut"


# every tile with whole tiles only, with cut ones only and with both (64 x 128: never both); rows, columns and K that are no
# whole tiles anywhere
@pytest.mark.parametrize("tile,kind,M,N,K", [
    ((64, 128), "whole", 43, 7, 72), ((64, 128), "cut", 70, 7, 2280),
    ((128, 128), "whole", 5529, 279, 136), ((128, 128), "cut", 1730, 7, 3896), ((128, 128), "mixed", 5950, 1295, 2016),
    ((128, 256), "whole", 5596, 655, 72), ((128, 256), "cut", 5424, 143, 2864), ((128, 256), "mixed", 796, 9583, 2016),
    ((256, 256), "whole", 804, 9503, 72), ((256, 256), "cut", 385, 5415, 5304), ((256, 256), "mixed", 1762, 9351, 936),
])
def test_linear_of_every_tile_whole_and_cut(hip, tile, kind, M, N, K):
    sums = torch.empty(hip.linear_scratch_bytes(M), dtype=torch.uint8, device=DEV)
    with_sums = gemm_kind(hip.linear_plan(M, N, K)) == (tile, kind)
    assert with_sums or gemm_kind(hip.linear_plan(M, N, K, scratch_bytes=0)) == (tile, kind)
    x, w = rnd(M, K, seed=90), rnd(N, K, seed=91, scale=K ** -0.5)
    want = (x.double() @ w.double().T).to(BF)
    y = torch.full((M + 1, N + 8), 5.0, dtype=BF, device=DEV)
    hip.linear(x, w, y[:M, :N], scratch=sums if with_sums else sums[:0])
    assert_close_ulp(y[:M, :N].contiguous(), want, what=f"{M} x {N} x {K}")
    assert (y[M:] == 5.0).all() and (y[:, N:] == 5.0).all()


@pytest.mark.parametrize("tile,kind,M,I,K", [
    ((64, 128), "whole", 43, 8, 72), ((64, 128), "cut", 70, 8, 2280),
    ((128, 128), "whole", 137, 5776, 136), ((128, 128), "cut", 1730, 8, 3896), ((128, 128), "mixed", 2409, 1696, 2232),
    ((128, 256), "whole", 203, 8312, 72), ((128, 256), "cut", 5999, 72, 3016), ((128, 256), "mixed", 545, 6600, 1960),
    ((256, 256), "whole", 529, 6640, 72), ((256, 256), "cut", 2747, 456, 5400), ((256, 256), "mixed", 5927, 1352, 1048),
])
def test_linear_swiglu_out_of_every_tile_whole_and_cut(hip, tile, kind, M, I, K):
    with_sums = gemm_kind(hip.linear_plan(M, 2 * I, K, True)) == (tile, kind)
    assert with_sums or gemm_kind(hip.linear_plan(M, 2 * I, K, True, 0)) == (tile, kind)
    check_swiglu_out(hip, M, I, K, hip.linear_scratch_bytes(M) if with_sums else 0)


@pytest.mark.parametrize("tile,kind,B,S,Hq,Hkv,hd,K", [
    ((64, 128), "cut", 5, 14, 1, 1, 8, 2280), ((128, 128), "whole", 3, 1843, 31, 2, 8, 136),
    ((128, 128), "cut", 5, 346, 1, 1, 8, 3896), ((128, 128), "mixed", 7, 850, 65, 8, 16, 2016),
    ((128, 256), "whole", 4, 1399, 37, 2, 16, 72), ((128, 256), "cut", 3, 1808, 14, 2, 8, 2864),
    ((128, 256), "mixed", 4, 199, 583, 8, 16, 2016), ((256, 256), "whole", 4, 201, 281, 8, 32, 72),
    ((256, 256), "cut", 5, 77, 661, 8, 8, 5304), ((256, 256), "mixed", 2, 881, 1153, 8, 8, 936),
])
def test_linear_rope_kv_of_every_tile_whole_and_cut(hip, tile, kind, B, S, Hq, Hkv, hd, K):
    M, N = B * S, (Hq + 2 * Hkv) * hd
    with_sums = gemm_kind(hip.linear_plan(M, N, K)) == (tile, kind)
    assert with_sums or gemm_kind(hip.linear_plan(M, N, K, scratch_bytes=0)) == (tile, kind)
    check_rope_kv(hip, B, S, Hq, Hkv, hd, K, hip.linear_scratch_bytes(M) if with_sums else 0)


# the tiles between (above 128 rows, whole k-tiles): halves of the rows that differ by a 16-row group per wave, last tiles of a few rows
@pytest.mark.parametrize("tile,kind,M,N,K", [
    ((160, 128), "whole", 650, 11017, 64), ((160, 128), "cut", 129, 3023, 2560), ((160, 256), "whole", 902, 8349, 1088),
    ((160, 256), "cut", 131, 10909, 3328), ((192, 128), "whole", 513, 8514, 256), ((192, 128), "cut", 164, 2809, 5184),
    ((192, 256), "whole", 1123, 8527, 192), ((192, 256), "cut", 169, 11013, 5056), ((192, 256), "mixed", 5166, 4666, 3968),
    ((224, 256), "whole", 1025, 10942, 192), ((224, 256), "cut", 193, 11270, 4928), ((224, 256), "mixed", 1293, 11992, 2176),
])
def test_linear_of_the_tiles_between(hip, tile, kind, M, N, K):
    test_linear_of_every_tile_whole_and_cut(hip, tile, kind, M, N, K)


@pytest.mark.parametrize("tile,kind,M,I,K", [
    ((160, 128), "whole", 652, 5480, 64), ((160, 128), "cut", 130, 1440, 2560), ((160, 256), "whole", 791, 4680, 384),
    ((160, 256), "cut", 259, 2696, 3456), ((192, 128), "whole", 514, 4904, 384), ((192, 128), "cut", 168, 1392, 5184),
    ((192, 256), "whole", 802, 5760, 320), ((192, 256), "cut", 170, 5464, 5760), ((224, 256), "whole", 1031, 5416, 896),
    ((224, 256), "cut", 193, 5488, 5056), ((224, 256), "mixed", 1314, 5960, 2368),
])
def test_linear_swiglu_out_of_the_tiles_between(hip, tile, kind, M, I, K):
    test_linear_swiglu_out_of_every_tile_whole_and_cut(hip, tile, kind, M, I, K)


@pytest.mark.parametrize("tile,kind,B,S,Hq,Hkv,hd,K", [
    ((160, 128), "whole", 2, 651, 357, 7, 16, 64), ((160, 128), "cut", 3, 45, 368, 2, 8, 2816), ((160, 256), "whole", 4, 388, 308, 4, 16, 1088),
    ((160, 256), "cut", 2, 134, 85, 1, 64, 3328), ((192, 128), "whole", 2, 322, 96, 6, 64, 256), ((192, 128), "cut", 3, 54, 520, 8, 8, 3584),
    ((192, 256), "whole", 3, 540, 732, 6, 8, 192), ((192, 256), "cut", 2, 282, 91, 7, 64, 5760), ((224, 256), "whole", 4, 645, 579, 1, 8, 256),
    ((224, 256), "cut", 2, 328, 54, 6, 64, 5696),
])
def test_linear_rope_kv_of_the_tiles_between(hip, tile, kind, B, S, Hq, Hkv, hd, K):
    test_linear_rope_kv_of_every_tile_whole_and_cut(hip, tile, kind, B, S, Hq, Hkv, hd, K)


@pytest.mark.parametrize("M,I,K", [(40, 1000, 2056), (128, 512, 4096), (300, 1000, 4104), (777, 2048, 4096)])
def test_linear_swiglu_out_pieces(hip, M, I, K):
    """[up; gate] pairs in cut tiles: the activation after the sums are complete."""
    check_swiglu_out(hip, M, I, K, hip.linear_scratch_bytes(M))


def check_swiglu_out(hip, M, I, K, sums_bytes):
    x, w1 = rnd(M, K, seed=92), rnd(2 * I, K, seed=93, scale=K ** -0.5)
    act, h = torch.empty(M, I, dtype=BF, device=DEV), torch.empty(M, 2 * I, dtype=BF, device=DEV)
    hip.linear_swiglu_out(x, w1, act, h, torch.empty(max(16, sums_bytes), dtype=torch.uint8, device=DEV)[:sums_bytes])
    u, g = (x.double() @ w1.double().T).to(BF).float().chunk(2, 1)
    want = ((g / (1 + torch.exp(-g))).to(BF).float() * u).to(BF)
    # up, gate and silu(gate) are each rounded: one step of any of them is at most 2^-7 of the result
    assert ((act.float() - want.float()).abs() <= 2.0 ** -7 * 3 * want.float().abs() + 2.0 ** -12).all()
    assert (ulp_diff(act, want) > 0).float().mean().item() < 0.05


@pytest.mark.parametrize("M,I,K", [(33, 17, 64), (64, 1000, 520), (512, 12288, 64), (1536, 4090, 136)])
def test_linear_swiglu_out_without_a_buffer_for_the_projection(hip, M, I, K):
    """Up to 64 rows, and from 192 tiles of 256 rows x 128 pairs on: any number of pairs, the same bits as with a buffer."""
    x, w1 = rnd(M, K, seed=96), rnd(2 * I, K, seed=97, scale=K ** -0.5)
    sums = torch.empty(max(16, hip.linear_scratch_bytes(M)), dtype=torch.uint8, device=DEV)
    got, want = (torch.full((M, I + 3), 5.0, dtype=BF, device=DEV) for _ in range(2))
    hip.linear_swiglu_out(x, w1, got[:, :I], sums=sums)
    hip.linear_swiglu_out(x, w1, want[:, :I], torch.empty(M, 2 * I, dtype=BF, device=DEV), sums)
    assert torch.equal(got, want) and (got[:, I:] == 5.0).all()
    u, g = (x.double() @ w1.double().T).to(BF).float().chunk(2, 1)
    ref = ((g / (1 + torch.exp(-g))).to(BF).float() * u).to(BF)
    assert ((got[:, :I].float() - ref.float()).abs() <= 2.0 ** -7 * 3 * ref.float().abs() + 2.0 ** -12).all()


@pytest.mark.parametrize("B,S,Hq,Hkv,hd,K", [(48, 1, 8, 2, 64, 4096), (1, 128, 8, 2, 64, 4096), (3, 100, 4, 1, 128, 4104), (2, 389, 16, 4, 128, 4096)])
def test_linear_rope_kv_pieces(hip, B, S, Hq, Hkv, hd, K):
    """The q/k/v projection in cut tiles, rotated and cached after the sums: the two calls on the same plan, bit for bit."""
    check_rope_kv(hip, B, S, Hq, Hkv, hd, K, hip.linear_scratch_bytes(B * S))


def check_rope_kv(hip, B, S, Hq, Hkv, hd, K, sums_bytes):
    N, Smax, start = (Hq + 2 * Hkv) * hd, S + 11, 5
    x, w = rnd(B * S, K, seed=94), rnd(N, K, seed=95, scale=K ** -0.5)
    sums = torch.empty(max(16, sums_bytes), dtype=torch.uint8, device=DEV)[:sums_bytes]
    pos = torch.arange(start, start + S, dtype=torch.int32, device=DEV)
    table = O.rope_table(start + S, hd, 500000, BF).to(DEV)
    out = [torch.empty(B * S, N, dtype=BF, device=DEV) for _ in range(2)]
    kc = [torch.zeros(B, Hkv, Smax, hd, dtype=BF, device=DEV) for _ in range(2)]
    vc = [torch.zeros_like(kc[0]) for _ in range(2)]
    hip.linear(x, w, out[0], scratch=sums)
    hip.rope_kv_write(out[0], table, False, pos, kc[0], vc[0], B, S, Hq, Hkv, hd)
    hip.linear_rope_kv(x, w, out[1], table, pos, kc[1], vc[1], B, S, Hq, Hkv, hd, sums)
    assert torch.equal(out[0], out[1]) and torch.equal(kc[0], kc[1]) and torch.equal(vc[0], vc[1])
    hip.raise_on_device_error(out[0].device)


def test_decode_batches_beyond_the_reach_of_the_gemm_stay_with_the_bands(hip):
    """A tile of 256 rows this far apart is out of the reach of a 2 GiB offset, 64 of them are not: with memory for partial
    sums or without, the weight-streaming kernel serves them, to the same bits."""
    M, K, ld = 40, 64, (1 << 22) + 8
    wide = torch.zeros((M - 1) * ld + K, dtype=BF, device=DEV)
    x = wide.as_strided((M, K), (ld, 1))
    x.copy_(rnd(M, K, seed=70))
    sums = torch.empty(1 << 20, dtype=torch.uint8, device=DEV)
    w = rnd(48, K, seed=71)
    plain, act = torch.empty(M, 48, dtype=BF, device=DEV), torch.empty(M, 24, dtype=BF, device=DEV)
    want, want_act = torch.empty_like(plain), torch.empty_like(act)
    hip.linear_multi((x.contiguous(), w, want, hip.EPI_NONE))
    hip.linear_multi((x.contiguous(), w, want_act, hip.EPI_SWIGLU))
    hip.linear(x, w, plain, scratch=sums)
    hip.linear_swiglu_out(x, w, act, sums=sums)
    assert torch.equal(plain, want) and torch.equal(act, want_act)
    kc, vc = (torch.zeros(M, 1, 8, 8, dtype=BF, device=DEV) for _ in range(2))
    pos, table = torch.tensor([3], dtype=torch.int32, device=DEV), O.rope_table(8, 8, 500000, BF).to(DEV)
    hip.linear_rope_kv(x, w, plain, table, pos, kc, vc, M, 1, 4, 1, 8, sums)
    hip.rope_kv_write(want, table, False, pos, *(torch.empty_like(kc) for _ in range(2)), M, 1, 4, 1, 8)
    assert torch.equal(plain, want) and torch.equal(vc[:, 0, 3], want[:, 40:])
    hip.raise_on_device_error(plain.device)


def quantised(w):
    """(e4m3 bytes, scales, the values they stand for in float64)"""
    scale = (w.float().abs().amax(1) / 448.0).clamp_min(2.0 ** -20).to(BF)
    w8 = (w.float() / scale.float()[:, None]).clamp(-448, 448).to(torch.float8_e4m3fn)
    return w8, scale


# bands of 2, 8, 9 (with a ragged last one), 16 and 32 columns; K within a chunk, ragged and of many chunks; the first and the last
# row counts of both input layouts
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("M,D,K1,K2", [(2, 264, 48, 1040), (8, 2048, 256, 272), (9, 2056, 1040, 48), (16, 4096, 512, 1552), (7, 8192, 1024, 3584),
                                       (12, 8192, 272, 1024)])
def test_linear_resid_and_the_projections_of_its_rows(hip, M, D, K1, K2, fp8):
    """Output projections with the residual updates, then a projection of the undivided rows they leave, each against the
    float64 product of what it was given: one bf16 step per rounding between input and result (sums of fp32 products are
    far closer than that), and the sums of squares to fp32 accuracy."""
    class Lin:
        pass
    dq = lambda l: l.weight.double() * l.scales.double()[:, None] if fp8 else l.weight.double()
    lins = []
    for i, K in enumerate((K1, K2)):
        l = Lin()
        l.weight = rnd(D, K, seed=120 + i, scale=K ** -0.5)
        if fp8:
            l.weight, l.scales = quantised(l.weight)
        lins.append(l)
    xs = [rnd(M, K, seed=122 + i) for i, K in enumerate((K1, K2))]
    gains = [rnd(D, seed=124 + i) * 0.1 + 1 for i in range(2)]
    resid0 = rnd(M, D, seed=126) * 4
    n = hip.linear_resid_sums(D)
    assert n == -(-D // (-(-D // 256)))
    a, m = (x.double() @ dq(l).T for x, l in zip(xs, lins))
    step = lambda t: 2.0 ** -8 * t.abs()          # half a bf16 step
    w, eps = rnd(512, D, seed=127, scale=D ** -0.5), 1e-5

    def project(x, sums, fold=None):
        y = torch.full((M, 516), 5.0, dtype=BF, device=DEV)
        hip.linear_multi((hip.Normed(x, sums, eps, fold), w, y[:, :512], hip.EPI_NONE))
        rs = torch.rsqrt(sums.double().sum(1, keepdim=True) / D + eps)
        want = x.double() @ w.double().T * rs
        assert ((y[:, :512].double() - want).abs() <= 1.01 * step(want) + 1e-5).all() and (y[:, 512:] == 5.0).all()
        return y

    for joint in (False, True):
        resid, outs = resid0.clone(), [torch.full((M, D), 7.0, dtype=BF, device=DEV) for _ in range(2)]
        sums = [torch.full((M, n), 7.0, device=DEV) for _ in range(2)]
        first = (xs[0], lins[0]) if joint else (xs[0], lins[0], gains[0], outs[0], sums[0])
        hip.linear_resid(first, (xs[1], lins[1], gains[1], outs[1], sums[1]), resid, joint=joint)
        r0, got = resid0.double(), resid.double()
        r1 = r0 + a
        want = r1 + m
        bound = (2 if fp8 else 1) * (step(a) + step(m)) + step(r1) + step(a + m) + step(want)    # (rounded before a scale too)
        assert ((got - want).abs() <= 1.05 * bound + 1e-4).all()
        assert torch.equal(outs[1], (got * gains[1].double()).to(BF))
        assert torch.allclose(sums[1].double().sum(1), got.square().sum(1), rtol=1e-5)
        if not joint:    # what the first update leaves is not stored: its rows to the same bounds
            assert ((outs[0].double() / gains[0].double() - r1).abs() <= 1.05 * (bound + step(r1)) + 1e-4).all()
            assert torch.allclose(sums[0].double().sum(1), r1.square().sum(1), rtol=2e-2)
        else:
            assert (outs[0] == 7.0).all() and (sums[0] == 7.0).all()
        total = torch.full((M, 1), 7.0, device=DEV)
        y = project(outs[1], sums[1], (sums[1], total))
        assert torch.allclose(total[:, 0].double(), sums[1].double().sum(1), rtol=1e-6)
        assert (ulp_diff(project(outs[1], total), y) <= 1).all()


def parts_of(x, count):
    """Sums of squares of `count` runs of columns, [M, count] fp32."""
    D = x.shape[1]
    runs = torch.zeros(x.shape[0], count, dtype=torch.float64, device=DEV)
    return runs.index_add_(1, torch.arange(D, device=DEV) * count // D, x.double().square()).float()


def rotated(t, table, hd):
    """Interleaved pairs of float64 heads [M, n] turned by table [hd / 2, 2]."""
    v, c, s = t.view(t.shape[0], -1, hd // 2, 2), table[:, 0].double(), table[:, 1].double()
    return torch.stack([v[..., 0] * c - v[..., 1] * s, v[..., 1] * c + v[..., 0] * s], -1).view_as(t)


# both input layouts of a band (to 8 rows, from 9), the e4m3 ones too; sums as one part, several and the most there may be; K of
# one chunk and of many, ragged bands
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("M,D,parts,parts2,Hq,Hkv,hd,I", [
    (3, 272, 17, 5, 4, 2, 64, 72), (8, 1024, 128, 256, 8, 1, 128, 456), (9, 2048, 256, 300, 8, 2, 64, 200), (13, 528, 511, 512, 4, 2, 64, 1000),
    (16, 8192, 256, 1, 8, 1, 128, 456), (16, 4096, 256, 256, 32, 8, 128, 1400)])
def test_every_projection_of_undivided_rows(hip, M, D, parts, parts2, Hq, Hkv, hd, I, fp8):
    """Rows whose root mean squares lie a factor of 64 apart, to be divided by the projection: q/k/v with the RoPE and cache
    epilogue and up/gate with the activation, in one launch, alone, and beside the attention on the sums that the q/k/v
    launch has added, each against float64.  A rounding moves a value by up to 2^-8 of it; fp32 sums are closer by far."""
    eps, N, Smax, pos = 1e-5, (Hq + 2 * Hkv) * hd, 64, 37
    spread = 2.0 ** ((torch.arange(M, device=DEV) * 5 % 7) - 3.0)
    x, x2 = ((rnd(M, D, seed=300 + i).double() * s[:, None]).to(BF) for i, s in enumerate((spread, spread.flip(0))))
    sums, sums2 = parts_of(x, parts), parts_of(x2, parts2)
    w, w2 = rnd(N, D, seed=302, scale=D ** -0.5), rnd(2 * I, D, seed=303, scale=D ** -0.5)
    table = O.rope_table(Smax, hd, 10000.0, BF).to(DEV)
    p = torch.tensor([pos], dtype=torch.int32, device=DEV)
    if fp8:
        (w, sc), (w2, sc2) = quantised(w), quantised(w2)
    step = lambda t: 2.0 ** -8 * t.abs()

    def product(x, sums, w, scales):
        """(x w^T of the divided rows, what its rounding and the fp32 sum may move it by)"""
        rs = torch.rsqrt(sums.double().sum(1, keepdim=True) / D + eps)
        f = 1.0 if scales is None else scales.double()
        v = (x.double() @ w.double().T) * rs * f
        return v, (1 if scales is None else 2) * step(v) + 2.0 ** -20 * (x.double().abs() @ w.double().abs().T) * rs * f

    v, dv = product(x, sums, w, sc if fp8 else None)
    n_qk, tab = (Hq + Hkv) * hd, table[pos].view(hd // 2, 2)
    pair = lambda t: t.view(M, -1, 2).flip(-1).reshape(M, -1)
    want_qk = rotated(v[:, :n_qk], tab, hd)
    want = torch.cat([want_qk, v[:, n_qk:]], 1)
    bound = torch.cat([dv[:, :n_qk] + pair(dv[:, :n_qk]) + step(want_qk), dv[:, n_qk:]], 1)
    (u, g), (du, dg) = (t.split(I, 1) for t in product(x2, sums2, w2, sc2 if fp8 else None))
    act = torch.nn.functional.silu(g)
    want_act, bound_act = act * u, u.abs() * (1.1 * dg + step(act)) + (act.abs() + 1.1 * dg) * du + step(act * u)

    def check(got, want, bound, what):
        assert ((got.double() - want).abs() <= 1.05 * bound + 1e-6).all(), what

    proj = lambda x, w, s, out, epi: (x, w, s, out, epi) if fp8 else (x, w, out, epi)
    multi = hip.linear_fp8_multi if fp8 else hip.linear_multi
    scales, scales2 = (sc, sc2) if fp8 else (None, None)
    for form in ("one launch", "beside", "alone"):
        qkv, out = torch.full((M, N), 5.0, dtype=BF, device=DEV), torch.full((M, I + 8), 5.0, dtype=BF, device=DEV)
        kc, vc = (rnd(M, Hkv, Smax, hd, seed=304 + i) for i in range(2))
        rope = hip.rope_kv_epilogue(table, p, kc, vc, Hq, Hkv, hd)
        total = torch.full((M, 1), 7.0, device=DEV)
        if form == "one launch":
            multi(proj(hip.Normed(x, sums, eps), w, scales, qkv, rope), proj(hip.Normed(x2, sums2, eps), w2, scales2, out[:, :I], hip.EPI_SWIGLU))
        else:
            multi(proj(hip.Normed(x, sums, eps, (sums2, total)), w, scales, qkv, rope))
            assert torch.allclose(total[:, 0].double(), sums2.double().sum(1), rtol=1e-6)
            up_gate = proj(hip.Normed(x2, total, eps), w2, scales2, out[:, :I], hip.EPI_SWIGLU)
            if form == "alone":
                multi(up_gate)
            else:
                scratch = torch.zeros(hip.attn_decode_scratch_bytes(M, Hq, hd, Smax) // 4, dtype=torch.float32, device=DEV)
                y, y1 = (torch.zeros(M, Hq * hd, dtype=BF, device=DEV) for _ in range(2))
                beside = hip.attn_decode_beside_fp8 if fp8 else hip.attn_decode_beside
                assert beside(qkv, kc, vc, p, y, scratch, M, Hq, Hkv, hd, up_gate)
                hip.attn_decode(qkv, kc, vc, p, y1, scratch, M, Hq, Hkv, hd)
                assert torch.equal(y, y1)
        got = torch.cat([qkv[:, :Hq * hd], kc[:, :, pos].reshape(M, -1), vc[:, :, pos].reshape(M, -1)], 1)
        check(got, want, bound, form + ": q, k, v")
        check(out[:, :I], want_act, bound_act, form + ": activation")
        assert (out[:, I:] == 5.0).all()
    hip.raise_on_device_error(x.device)


def test_undivided_rows_that_no_launch_serves_are_refused(hip):
    """Sums for a later launch of more rows than the projection has bands: nothing is launched."""
    x, y, sums, total = rnd(8, 64, seed=310), torch.full((8, 28), 5.0, dtype=BF, device=DEV), torch.ones(8, 2, device=DEV), torch.full((8, 1), 7.0, device=DEV)
    with pytest.raises(hip.LadderHipError):
        hip.linear_multi((hip.Normed(x, sums, 1e-5, (sums, total)), rnd(28, 64, seed=311), y, hip.EPI_NONE))
    torch.cuda.synchronize()
    assert (y == 5.0).all() and (total == 7.0).all()
