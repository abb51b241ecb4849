"""The attention of a prefill batch (head dim 256, more than a window of positions: scores in one launch,
the chunks of 32 keys folded per row in another), bit-exact against the same positions in windows of 8:
query counts around the least that takes it (96 at 24 heads), ragged row tiles, prefixes around a chunk's and
a tile's edge, group sizes 1, 2, 8 and 12, both score tiles (64 wide, and 128 where those are 768 or more: 256
queries of 24 heads over 2048 keys), the last keys that a cache of 2048 holds, and keys whose scores are
infinite or NaN (such a chunk adds nothing to any query that sees it)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from gpu_util import dev, empty_bf16, host, need_gpu, rand_bf16, write_device  # noqa: E402


@pytest.fixture(scope="module")
def ctx():
    need_gpu()
    import mtpx
    c = mtpx.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("HQ,HK,pre,n,odd", [
    (24, 2, 0, 96, False), (24, 2, 31, 95, False), (24, 24, 33, 97, False), (12, 12, 127, 193, False),
    (32, 4, 96, 73, False), (12, 1, 1792, 256, False), (24, 2, 1663, 256, False), (24, 2, 1792, 256, False),
    (24, 2, 1900, 148, False), (24, 2, 40, 101, True),
    (16, 8, 257, 200, True)])
def test_attention_batch_matches_windows(ctx, HQ, HK, pre, n, odd):
    import mtpx
    layer = dict(hidden=256, experts=16, top_k=4, expert_width=128, group_size=32, heads=HQ, kv_heads=HK,
                 head_dim=256, rot_dims=64, index_dim=32, rope_theta=1e7, eps=1e-6, max_positions=2048)
    hc, V = 4, 1000
    head = mtpx.MTPHead(ctx, mtpx.HeadConfig(mtpx.LayerConfig(**layer), hc, 64, V, 500, 980), seed=23)
    W = hc * layer["hidden"]
    r = np.random.default_rng(1000 * HQ + pre + n)
    kc, vc = np.zeros((HK, 2048, 256), np.uint16), np.zeros((HK, 2048, 256), np.uint16)
    kc[:, :pre] = rand_bf16(r, (HK, pre, 256))
    vc[:, :pre] = rand_bf16(r, (HK, pre, 256))
    if odd:
        kc[0, 3, 5] = 0x7fc0            # a NaN key: every score of it is NaN
        kc[HK - 1, 35] = 0x7f7f         # keys at the format's limit: scores of either sign overflow
        kc[HK - 1, 36] = 0xff7f
    ids, multi = dev(r.integers(0, V, n).astype(np.int32)), dev(rand_bf16(r, (n, W)))
    caches = []
    for _ in range(2):
        kv = mtpx.KVCache(ctx, HK, 256, 2048)
        kp, vp, _ = kv.buffers()
        write_device(kp, kc)
        write_device(vp, vc)
        kv.offset = pre
        caches.append(kv)
    print("case attention batch", HQ, HK, pre, n, odd, flush=True)
    got, want = empty_bf16(n, W), empty_bf16(n, W)
    head.forward(caches[0], ids, multi, got)
    for w0 in range(0, n, 8):
        w1 = min(n, w0 + 8)
        head.forward(caches[1], ids[w0:w1], multi[w0:w1], want[w0:w1])
    assert np.array_equal(host(got), host(want))
    for kv in caches:
        kv.close()
    head.close()
