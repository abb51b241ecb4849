"""GPU parity of the batch GEMMs (csrc/gemm.hip), bit-exact: every depth they take at the edges of their
row blocks and 16-token tiles against the oracle, inputs outside the plain walk's exponent range (blocks
above 4096, denormal and zero blocks, infinities), checkpoint rows that their loads do not take, and the
expert chunks against the verify path's windows, with ordinary and with large activations."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from gpu_util import dev, empty_bf16, host, need_gpu, qweights, rand_bf16, read_device, write_device  # noqa: E402
from oracle import oracle as O  # noqa: E402


@pytest.fixture(scope="module")
def ctx():
    need_gpu()
    import mtpx
    c = mtpx.Context(0)
    yield c
    c.close()


def _check(ctx, wq, s, b, gs, x, ds=None, db=None, gemm=True, packed=False):
    """gemm: whether the batch GEMM (which prepares x in limb form) is what runs."""
    M, N = x.shape[0], wq.shape[0]
    y_o, yf_o = O.qmv(wq, s, b, gs, x)
    ds, db = dev(s) if ds is None else ds, dev(b) if db is None else db
    y, yf = empty_bf16(M, N), torch.zeros(M, N, dtype=torch.float32, device="cuda")
    sb = ctx.pack_sb(ds, db, x.shape[1], gs) if packed else None
    ctx.profile(True)
    ctx.profile_reset()
    ctx.qmv(dev(wq), ds, db, gs, dev(x), y, yf, sb=sb)
    launched = ctx.profile_stats()
    ctx.profile(False)
    assert ("xlimb" in launched) == gemm, launched
    assert np.array_equal(host(yf).view(np.uint32), yf_o.view(np.uint32))
    assert np.array_equal(host(y), y_o)


# row blocks of 128 (K 2560), 64 (6144), 32 (8192, 10240) and 256 (320) rows; tiles of 16 tokens; the fewest tokens or
# rows that it takes at each depth
@pytest.mark.parametrize("N,K,gs,M", [
    (1, 2560, 64, 301), (127, 2560, 32, 304), (128, 2560, 64, 305), (385, 2560, 64, 325), (17, 2560, 32, 319),
    (5121, 2560, 64, 9), (5247, 2560, 32, 16), (5120, 2560, 64, 25),
    (64, 6144, 64, 257), (641, 6144, 32, 64), (5121, 6144, 32, 9), (1, 10240, 32, 257), (325, 10240, 64, 81),
    (5150, 10240, 64, 17), (31, 8192, 64, 129), (200, 8192, 32, 52), (254, 320, 64, 9), (513, 320, 32, 47),
    (16, 320, 64, 16),
])
def test_gemm_edges_bit_exact(ctx, N, K, gs, M):
    print("case", N, K, gs, M, flush=True)
    r = np.random.default_rng(N * 7 + K + M)
    wq, s, b = qweights(r, N, K, gs)
    _check(ctx, wq, s, b, gs, rand_bf16(r, (M, K)))


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("N,K,gs,M", [
    (385, 2560, 64, 300), (5120, 2560, 32, 24), (65, 6144, 32, 256), (640, 6144, 64, 64), (33, 10240, 64, 256),
    (325, 10240, 64, 80), (31, 8192, 64, 128), (200, 8192, 32, 51), (324, 10240, 64, 9), (255, 320, 64, 9)])
def test_batch_by_windows_below_the_gemms_line(ctx, N, K, gs, M, packed):
    """The most tokens that the windows take, a mixer's rows at nine tokens, and an odd count of scales, which its loads do
    not take: the GEMV's windows."""
    print("case windows", N, K, gs, M, packed, flush=True)
    r = np.random.default_rng(N + K + M)
    wq, s, b = qweights(r, N, K, gs)
    _check(ctx, wq, s, b, gs, rand_bf16(r, (M, K)), gemm=False, packed=packed)


@pytest.mark.parametrize("K,gs", [(2560, 64), (6144, 32), (10240, 64), (320, 32)])
def test_gemm_extreme_blocks_bit_exact(ctx, K, gs):
    """Tiles with and without a token above 4096 side by side, blocks of every size between 2^-120 and 2^100,
    zero blocks, and an infinity (whose block value the quantiser defines as any other exponent)."""
    print("case", K, gs, flush=True)
    r = np.random.default_rng(K)
    wq, s, b = qweights(r, 70, K, gs)
    x = r.standard_normal((310, K)).astype(np.float32)
    x[5, 32:64] *= 3e4                                            # the first tile walks with the factor
    x[17] *= np.float32(2.0) ** np.repeat(np.linspace(-118, -2, K // 32).astype(int), 32)
    x[18] = 0
    x[19, ::2] *= 1e-7
    x[36] *= np.float32(2.0) ** np.repeat(np.linspace(0, 90, K // 32).astype(int), 32)
    xb = O.f32_to_bf16(x)
    xb[37, 64] = 0x7f80
    _check(ctx, wq, s, b, gs, xb)


def test_gemm_past_two_gib_of_weights(ctx):
    """A matrix of more than 2^31 bytes, bit-equal to a window of 8 and a token more, rows of both ends included."""
    N, K, gs, M = 1677760 + 5, 2560, 64, 9
    g = torch.Generator(device="cuda").manual_seed(7)
    wq = torch.randint(-2 ** 31, 2 ** 31 - 1, (N, K // 8), generator=g, device="cuda", dtype=torch.int32)
    s, b = ((torch.rand(N, K // gs, generator=g, device="cuda") * f).bfloat16() for f in (0.01, -0.08))
    x = dev(rand_bf16(np.random.default_rng(3), (M, K)))
    y, want = empty_bf16(M, N), empty_bf16(M, N)
    print("case two GiB", N, K, flush=True)
    ctx.profile(True)
    ctx.profile_reset()
    ctx.qmv(wq, s, b, gs, x, y)
    launched = ctx.profile_stats()
    ctx.profile(False)
    ctx.qmv(wq, s, b, gs, x[:8], want[:8])
    ctx.qmv(wq, s, b, gs, x[8:], want[8:])
    ctx.synchronize()
    assert "xlimb" in launched, launched
    assert torch.equal(y.view(torch.int16), want.view(torch.int16))


def _odd(a):
    """The bf16 bits a on the device, from an odd element on."""
    p = torch.zeros(a.size + 1, dtype=torch.bfloat16, device="cuda")
    p[1:] = dev(a).reshape(-1)
    return p[1:].view(*a.shape)


def test_gemm_two_byte_aligned_scales(ctx):
    """Scales and biases at an odd bf16 offset, or one of them: copied for the call."""
    r = np.random.default_rng(2)
    wq, s, b = qweights(r, 48, 2560, 64)
    x = rand_bf16(r, (310, 2560))
    _check(ctx, wq, s, b, 64, x, _odd(s), _odd(b))
    _check(ctx, wq, s, b, 64, x, dev(s), _odd(b))
    _check(ctx, wq, s, b, 64, x[:21], _odd(s), _odd(b), gemm=False)


def test_adopted_two_byte_aligned_scales(ctx):
    """A head adopted with every scale and bias array of its batch matrices at an odd bf16 offset takes the same launches as
    one with aligned arrays, and gives the same bits."""
    import mtpx
    lc = mtpx.LayerConfig(2560, 24, 4, 640, 64, 24, 2, 256, 64, 128, 1e7, 1e-6, 256)
    cfg = mtpx.HeadConfig(lc, 4, 320, 1000, 500, 980)
    base = mtpx.MTPHead(ctx, cfg, seed=51)
    w, keep = base.weights(), []

    def odd(obj, prefix, rows, k):
        for part in "sb":
            a = read_device(getattr(obj, prefix + part), rows * (k // 64) * 2, np.uint16)
            keep.append(_odd(a))
            setattr(obj, prefix + part, keep[-1].data_ptr())

    H, W, E, F = 2560, 4 * 2560, 24, 640
    odd(w.layer, "qkv_", w.layer.qkv_rows, H)
    odd(w.layer, "o_", H, 24 * 256)
    for name, rows, k in (("gate_", E * F, H), ("up_", E * F, H), ("down_", E * H, F), ("sh_gate_", F, H),
                          ("sh_up_", F, H), ("sh_down_", H, F)):
        odd(w.layer.moe, name, rows, k)
    for q, rows, k in ((w.fc_embedding, H, H), (w.fc_hidden, H, H)):
        odd(q, "", rows, k)
    for m in (w.attn_hc, w.mlp_hc, w.final_hc):
        odd(m.down, "", 320, W)
        odd(m.up, "", W, 320)
        if m.inject.w:
            odd(m.inject, "", 4, W)
    head = mtpx.MTPHead.adopt(ctx, cfg, w)
    n = 90
    r = np.random.default_rng(n)
    ids, multi = dev(r.integers(0, 1000, n).astype(np.int32)), dev(rand_bf16(r, (n, W)))
    print("case adopted odd scales", flush=True)
    got = []
    for h in (base, head):
        kv = mtpx.KVCache(ctx, 2, 256, 256)
        out = empty_bf16(n, W)
        ctx.profile(True)
        ctx.profile_reset()
        h.forward(kv, ids, multi, out)
        got.append((host(out), {k: v[0] for k, v in ctx.profile_stats().items()}))
        ctx.profile(False)
        kv.close()
    head.close()
    base.close()
    assert got[0][1] == got[1][1]
    assert np.array_equal(got[0][0], got[1][0])


@pytest.mark.parametrize("gs,n,large", [(64, 200, False), (64, 200, True), (32, 149, False), (32, 149, True),
                                        (64, 1100, False)])
def test_expert_chunks_match_windows(ctx, gs, n, large):
    """A prompt whose experts run by chunks of 16 slots gives the verify windows' bits, and so does a window after it; large:
    the MoE's input scaled so that its blocks and the experts' activations pass 4096; 1100: a batch of 1024 positions and
    one of 76 behind it, every kernel of a long prompt at the model's widths."""
    import mtpx
    lc = mtpx.LayerConfig(2560, 96, 6, 640, gs, 24, 2, 256, 64, 128, 1e7, 1e-6, n + 8)
    cfg = mtpx.TargetConfig(lc, 16, 48, 4, 2, 4, 4, 320, 4000)
    cfg.ple_layer = -1
    t = mtpx.Target(ctx, cfg, seed=77)
    if large:
        sc = O.f32_to_bf16(np.full(4 * 2560, 1e5, np.float32))
        for i in range(2):
            write_device(t.layer_weights(i).mlp_hc.norm_scale, sc)
    ids = dev(np.random.default_rng(n).integers(0, 4000, n).astype(np.int32))
    print("case chunks", gs, n, large, flush=True)
    a, b = mtpx.TargetState(ctx, t), mtpx.TargetState(ctx, t)
    lg, mt = empty_bf16(4000), empty_bf16(n, 4 * 2560)
    t.prefill(a, ids, lg, mt)
    want = []
    for w in ids.split(8):
        lw, mw = empty_bf16(len(w), 4000), empty_bf16(len(w), 4 * 2560)
        t.verify(b, w.contiguous(), lw, mw)
        b.commit(len(w))
        want.append(host(mw))
    assert np.array_equal(host(mt), np.concatenate(want))
    assert np.array_equal(host(lg), host(lw)[-1])
    nxt, la, lb = dev(np.array([5, 6, 7, 8], np.int32)), empty_bf16(4, 4000), empty_bf16(4, 4000)
    t.verify(a, nxt, la)
    t.verify(b, nxt, lb)
    assert np.array_equal(host(la), host(lb))
    a.close()
    b.close()
    t.close()
