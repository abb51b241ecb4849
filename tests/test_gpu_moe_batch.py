"""The MoE block of a prefill batch (its own router launch, one expert order for all its tokens), bit-exact against the
same positions in windows of 8: one position more than a window, a tail that is no window, expert counts that do not
fill a wave's or a workgroup's rows, the largest counts, every instance of the router launch (by the 16-byte chunks of a
row: up to 128, up to 256, 320, more; whole and ragged), and the shared expert's gate as a bf16 row and as a q4 row."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from gpu_util import dev, empty_bf16, host, need_gpu, rand_bf16  # noqa: E402


@pytest.fixture(scope="module")
def ctx():
    need_gpu()
    import mtpx
    c = mtpx.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("H,E,K,n,q4", [
    (512, 16, 4, 9, False), (544, 1024, 16, 37, True), (1024, 31, 1, 255, False), (2048, 33, 3, 13, True),
    (1056, 40, 7, 20, False), (2080, 70, 5, 21, False), (4096, 16, 2, 33, False), (2560, 33, 3, 13, True),
    (2560, 520, 10, 30, False), (2560, 16, 10, 70, False)])
def test_moe_batch_matches_windows(ctx, H, E, K, n, q4):
    import mtpx
    layer = dict(hidden=H, experts=E, top_k=K, expert_width=128, group_size=32, heads=4, kv_heads=2, head_dim=64,
                 rot_dims=16, index_dim=32, rope_theta=1e7, eps=1e-6, max_positions=256)
    hc, V = 4 if H < 2048 or H == 2560 else 1, 1000
    cfg = mtpx.HeadConfig(mtpx.LayerConfig(**layer), hc, 64, V, 500, 980)
    head = mtpx.MTPHead(ctx, cfg, seed=31 + n)
    r = np.random.default_rng(E + n)
    used = head
    if q4:
        w = head.weights()
        row = [dev(r.integers(0, 2 ** 32, (1, H // 8), dtype=np.uint32).view(np.int32)),
               dev(rand_bf16(r, (1, H // 32), 0.01)), dev(rand_bf16(r, (1, H // 32), 0.05))]
        m = w.layer.moe
        m.shared_gate, m.shared_gate_sb = None, None
        m.shared_gate_w, m.shared_gate_s, m.shared_gate_b = (t.data_ptr() for t in row)
        used = mtpx.MTPHead.adopt(ctx, cfg, w)
    W = hc * H
    ids, multi = dev(r.integers(0, V, n).astype(np.int32)), dev(rand_bf16(r, (n, W)))
    kva, kvb = (mtpx.KVCache(ctx, 2, 64, 256) for _ in range(2))
    print("case MoE batch", H, E, K, n, q4, flush=True)
    got, want = empty_bf16(n, W), empty_bf16(n, W)
    ctx.profile(True)
    ctx.profile_reset()
    used.forward(kva, ids, multi, got)
    launched = ctx.profile_stats()
    ctx.profile(False)
    assert launched["moe_route_batch"][0] == 1, launched
    for w0 in range(0, n, 8):
        w1 = min(n, w0 + 8)
        used.forward(kvb, ids[w0:w1], multi[w0:w1], want[w0:w1])
    assert np.array_equal(host(got), host(want))
    kva.close()
    kvb.close()
    if used is not head:
        used.close()
    head.close()


# row blocks of 128 rows of H: whole ones and a last one of 32 rows; both sides of 1.25 slots per expert and of 200000
# output elements in all
@pytest.mark.parametrize("H,E,K,n,gs,chunks", [
    (1024, 32, 4, 70, 64, 1), (544, 16, 3, 100, 32, 1), (512, 9, 9, 45, 64, 1), (1024, 256, 8, 40, 32, 1),
    (1024, 256, 8, 39, 32, 0), (1024, 32, 4, 40, 64, 1), (1024, 32, 4, 39, 64, 0), (2560, 96, 6, 19, 64, 0)])
def test_expert_down_chunks_at_other_hidden_sizes(ctx, H, E, K, n, gs, chunks):
    """The expert down GEMM at expert width 640 takes any hidden size, where experts hold enough slots (it reads the
    experts' activations in limb form: its number of passes tells), bit-equal to windows of 8."""
    import mtpx
    lc = mtpx.LayerConfig(H, E, K, 640, gs, 4, 2, 64, 16, 32, 1e7, 1e-6, 256)
    head = mtpx.MTPHead(ctx, mtpx.HeadConfig(lc, 4, 64, 1000, 500, 980), seed=41 + n)
    W = 4 * H
    r = np.random.default_rng(H + n)
    ids, multi = dev(r.integers(0, 1000, n).astype(np.int32)), dev(rand_bf16(r, (n, W)))
    kva, kvb = (mtpx.KVCache(ctx, 2, 64, 256) for _ in range(2))
    print("case expert down", H, E, K, n, gs, flush=True)
    got, want = empty_bf16(n, W), empty_bf16(n, W)
    ctx.profile(True)
    ctx.profile_reset()
    head.forward(kva, ids, multi, got)
    launched = ctx.profile_stats()
    ctx.profile(False)
    assert launched["moe_route_batch"][0] == 1, launched
    if H != 2560:  # no projection here is of a depth that the dense GEMM takes
        assert launched.get("xlimb", (0,))[0] == chunks, launched
    for w0 in range(0, n, 8):
        w1 = min(n, w0 + 8)
        head.forward(kvb, ids[w0:w1], multi[w0:w1], want[w0:w1])
    assert np.array_equal(host(got), host(want))
    kva.close()
    kvb.close()
    head.close()
