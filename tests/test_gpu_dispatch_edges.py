"""GPU parity at the edges of the launch rules: the sizes where a kernel's split of the work has a
remainder, is smallest or largest, or hands over to another kernel."""
import numpy as np
import pytest

from cwick_amd import synth
from tests.conftest import assert_close

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)


@pytest.mark.parametrize("nh,batch,nope,rope,vdim", [(1, 1, 1, 0, 1), (3, 4, 127, 64, 31), (2, 5, 128, 64, 128),
                                                      (5, 3, 129, 8, 130), (2, 9, 300, 64, 192),
                                                      (4, 2, 512, 0, 65), (3, 2, 64, 17, 9), (2, 6, 448, 64, 8)])
def test_absorb_expand_edges(hip, orc, nh, batch, nope, rope, vdim):
    """Row counts around the 128 that a workgroup holds at a time, batches around its four queries."""
    import torch
    say("[case] absorb / expand", nh, batch, nope, rope, vdim)
    q_dim, kv_dim, kv_lora = nope + rope, nope + vdim, 512
    g = synth.rng(77)
    kvb = synth.f32_to_bf16(g.standard_normal((nh * kv_dim, kv_lora), dtype=np.float32))
    q = g.standard_normal((batch, nh, q_dim), dtype=np.float32)
    cacc = g.standard_normal((batch, nh, kv_lora), dtype=np.float32)
    s = torch.cuda.current_stream().cuda_stream
    d_kvb, d_q, d_c = torch.from_numpy(kvb.view(np.int16)).cuda(), torch.from_numpy(q).cuda(), torch.from_numpy(cacc).cuda()
    d_qabs = torch.zeros((batch, nh, synth.KDIM), dtype=torch.int16, device="cuda")
    d_out = torch.zeros((batch, nh, vdim), dtype=torch.float32, device="cuda")
    hip.mla_absorb_dev(d_kvb, d_q, nh * q_dim, batch, nh, q_dim, nope, rope, kv_dim, kv_lora, d_qabs, s)
    hip.mla_expand_dev(d_kvb, d_c, batch, nh, nope, vdim, kv_dim, kv_lora, d_out, s)
    torch.cuda.synchronize()
    for y in range(batch):
        ref = orc.mla_absorb(kvb, q[y], nope, rope, kv_dim)
        got = synth.bf16_to_f32(d_qabs[y].cpu().numpy().view(np.uint16))
        top = np.abs(ref).max()
        assert np.abs(got - ref).max() <= 2.0 ** -8 * top + 1e-4 * top, "absorb, query %d" % y
        assert np.array_equal(got[:, 512:512 + rope], synth.bf16_to_f32(synth.f32_to_bf16(q[y][:, nope:])))
        assert (got[:, 512 + rope:] == 0).all()
        ref = orc.mla_expand(kvb, cacc[y], nope, vdim, kv_dim)
        assert np.abs(d_out[y].cpu().numpy() - ref).max() <= 1e-4 * np.abs(ref).max(), "expand, query %d" % y


@pytest.mark.parametrize("n,pos0,nh,nkv", [
    (1, 4000, 16, 4),        # one position, its block's keys in slices
    (65, 4127, 16, 4),       # two blocks, the second of one position; slices end on and off the diagonal tile
    (70, 3990, 8, 8),        # one head per kv head: the diagonal is nine tiles wide
    (300, 700, 16, 4),       # blocks on either side of the two-term weights' 1024 keys
    (130, 5000, 16, 2),      # eight heads per kv head
    (33, 0, 16, 4),          # nothing to split
    (16, 16001, 16, 4),      # sixty slices and more: batches of sixteen in the merge, the last one short
    (16, 1100, 16, 4),       # more than eight slices, fewer than sixteen
])
def test_gqa_prefill_slices(hip, orc, n, pos0, nh, nkv):
    """Chunks whose position blocks do not fill the chip: the keys of a block in several slices."""
    say("[case] gqa prefill slices", n, pos0, nh, nkv)
    c = synth.cfg2_gqa_prefill(n, nh, nkv, 256, pos0, seed=78)
    cache = hip.KVCache(pos0 + n, nkv, 256)
    cache.write(0, c["k"].reshape(pos0 + n, -1), c["v"].reshape(pos0 + n, -1))
    got = hip.gqa_prefill(cache, pos0, c["q"], c["scale"])
    ref = orc.gqa_prefill(c["q"], c["k"], c["v"], pos0, c["scale"], nthreads=0)
    assert_close(got, ref, "gqa prefill slices", strict=pos0 >= 200)
    cache.free()


@pytest.mark.parametrize("n,pos0,nh,nkv", [
    (16, 0, 16, 4),          # one workgroup for each kv head, all its rows live
    (17, 2000, 16, 4),       # a second block of one position; slices
    (9, 1015, 16, 2),        # eight heads: blocks of eight positions on either side of the 1024 keys
    (65, 1500, 8, 8),        # one head: blocks of 64 positions, the second of one
    (600, 4000, 16, 4),      # more rows than that
])
def test_gqa_prefill_small_problems(hip, orc, n, pos0, nh, nkv):
    """Problems that do not fill the chip: blocks of 64 rows, whole and in slices, with a key that outgrows every
    reference before it (the tiles that follow the maximum)."""
    say("[case] gqa prefill, small problems", n, pos0, nh, nkv)
    c = synth.cfg2_gqa_prefill(n, nh, nkv, 256, pos0, seed=80)
    k = synth.bf16_to_f32(c["k"])
    late = (pos0 + n) * 2 // 3
    if pos0:
        k[late] = 30.0 * synth.bf16_to_f32(c["q"])[n - 1].reshape(nkv, nh // nkv, 256)[:, 0]
    k = synth.f32_to_bf16(k)
    cache = hip.KVCache(pos0 + n, nkv, 256)
    cache.write(0, k.reshape(pos0 + n, -1), c["v"].reshape(pos0 + n, -1))
    got = hip.gqa_prefill(cache, pos0, c["q"], c["scale"])
    ref = orc.gqa_prefill(c["q"], k, c["v"], pos0, c["scale"], nthreads=0)
    assert_close(got, ref, "gqa prefill, small problems", strict=False)
    cache.free()


@pytest.mark.parametrize("n,pos0,nh,nkv", [
    (1, 0, 16, 4), (31, 0, 16, 2), (32, 0, 4, 2),       # one tile: every wave scores it, a quarter of the dims each
    (33, 0, 16, 4),                                     # one tile for the first blocks, two for the last
    (70, 0, 8, 8), (97, 0, 16, 4), (129, 0, 16, 2),     # three, four and five tiles; diagonals of three tiles
    (64, 192, 16, 4), (63, 1, 8, 8),                    # blocks that end at and before a tile's border
    (1025, 0, 16, 4), (1060, 0, 8, 8),                  # two-term weights and plain ones, more than one round of blocks
    (40, 4000, 8, 8), (24, 2500, 4, 2),                 # slices, some of fewer tiles than waves
    (64, 1000, 16, 4), (237, 627, 16, 4),               # slices of a single tile
])
@pytest.mark.parametrize("late", [False, True])
def test_gqa_prefill_four_waves_a_block(hip, orc, n, pos0, nh, nkv, late):
    """Workgroups whose four waves share a block of 64 rows; with a key that outgrows every reference before it,
    for which the waves that meet it start over."""
    say("[case] gqa prefill, four waves a block", n, pos0, nh, nkv, late)
    c = synth.cfg2_gqa_prefill(n, nh, nkv, 256, pos0, seed=81)
    k = c["k"]
    if late:
        k = synth.bf16_to_f32(k)
        k[(pos0 + n) * 2 // 3] = 30.0 * synth.bf16_to_f32(c["q"])[n - 1].reshape(nkv, nh // nkv, 256)[:, 0]
        k = synth.f32_to_bf16(k)
    cache = hip.KVCache(pos0 + n, nkv, 256)
    cache.write(0, k.reshape(pos0 + n, -1), c["v"].reshape(pos0 + n, -1))
    got = hip.gqa_prefill(cache, pos0, c["q"], c["scale"])
    ref = orc.gqa_prefill(c["q"], k, c["v"], pos0, c["scale"], nthreads=0)
    assert_close(got, ref, "gqa prefill, four waves a block", strict=pos0 >= 200 and not late)
    cache.free()


@pytest.mark.parametrize("HD,rotary", [(256, 256), (256, 36), (128, 24), (128, 6)])
def test_gqa_prepare_head_sizes(hip, orc, HD, rotary):
    """The rotation over all and a part of a head, its halves in fours (four dims a lane) and not."""
    import torch
    say("[case] gqa prepare", HD, rotary)
    n, pos0, H, KV, eps = 3, 7, 5, 2, 1e-6
    g = synth.rng(HD)
    cos_t, sin_t = orc.build_rope(pos0 + n, rotary, 1e6)
    qp, kp, vp = (g.standard_normal((n, h * HD), dtype=np.float32) for h in (H, KV, KV))
    qn, kn = (g.standard_normal(HD, dtype=np.float32) * np.float32(0.1) for _ in range(2))
    d = lambda a: torch.from_numpy(a).cuda()
    ops = [d(a) for a in (qp, kp, vp, qn, kn, cos_t, sin_t)]
    q = torch.zeros((n, H, HD), dtype=torch.int16, device="cuda")
    cache = hip.KVCache(pos0 + n, KV, HD)
    q_ref, k_ref, v_ref = orc.gqa_prepare(qp, HD, kp, vp, pos0, H, KV, HD, qn, kn, eps, cos_t, sin_t, rotary)
    hip.gqa_prepare_dev(ops[0], HD, ops[1], ops[2], n, pos0, H, KV, HD, ops[3], ops[4], eps, ops[5], ops[6], rotary, q, cache,
                        torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    k_got, v_got = cache.read(pos0, n)
    assert np.array_equal(v_got.reshape(-1), v_ref.reshape(-1))
    for got, ref, h in ((q.cpu().numpy().view(np.uint16), q_ref, H), (k_got, k_ref, KV)):
        gf, rf = (synth.bf16_to_f32(x.reshape(n, h, HD)) for x in (got, ref))
        assert (np.abs(gf - rf) <= 2.0 ** -7 * np.abs(rf).max(axis=-1, keepdims=True)).all()
    cache.free()


def test_gqa_prefill_slices_late_maximum(hip, orc):
    """A key far along that beats everything before it: the slices' references differ by more than
    a slice's own weights may exceed its reference."""
    n, pos0, nh, nkv = 20, 3000, 16, 4
    c = synth.cfg2_gqa_prefill(n, nh, nkv, 256, pos0, seed=79)
    k = synth.bf16_to_f32(c["k"])
    k[2100] = 30.0 * synth.bf16_to_f32(c["q"])[0].reshape(nkv, nh // nkv, 256)[:, 0]
    k = synth.f32_to_bf16(k)
    cache = hip.KVCache(pos0 + n, nkv, 256)
    cache.write(0, k.reshape(pos0 + n, -1), c["v"].reshape(pos0 + n, -1))
    got = hip.gqa_prefill(cache, pos0, c["q"], c["scale"])
    ref = orc.gqa_prefill(c["q"], k, c["v"], pos0, c["scale"], nthreads=0)
    assert_close(got, ref, "gqa prefill slices, late maximum", strict=False)
    cache.free()


@pytest.mark.parametrize("nh,nkv,hd", [(16, 4, 256), (32, 4, 256), (16, 1, 256), (2, 2, 128), (4, 2, 128), (8, 2, 128),
                                       (64, 8, 128), (64, 4, 128)])
@pytest.mark.parametrize("n_keys", [1, 15, 64, 192, 193, 2049])
def test_gqa_decode_edges(hip, orc, n_keys, nh, nkv, hd):
    """Every group size of both head widths (the value product differs with them) at lengths around
    a tile, a workgroup's step, and the single-workgroup limit."""
    say("[case] gqa decode edges", n_keys, nh, nkv, hd)
    c = synth.cfg1_gqa_decode(n_keys, nh, nkv, hd, seed=80 + n_keys)
    cache = hip.KVCache(n_keys, nkv, hd)
    cache.write(0, c["k"], c["v"])
    got = hip.gqa_decode(cache, n_keys, c["q"], c["scale"])
    ref = orc.gqa_decode(c["q"], c["k"], c["v"], c["scale"], nthreads=0)
    err = np.abs(got - ref).max() / np.abs(ref).max()
    assert err < 2e-5, "rel %.2e" % err           # fp32 sums of exact products: nothing is rounded on the way
    cache.free()


@pytest.mark.parametrize("n_keys,nh,nkv,hd", [
    (4161, 64, 8, 128),      # 66 steps for 22 workgroups a kv head, a key in the last
    (8193, 16, 4, 256),      # 129 for 43
    (8256, 8, 4, 128),       # 129 whole ones for 43
    (700, 64, 64, 128),      # 11 for 4: one of them has a step less, and their last workgroup merges
])
def test_gqa_decode_steps_in_turn(hip, orc, n_keys, nh, nkv, hd):
    """Several steps per workgroup, dealt in turn: as many for each, one less for some, one that ends in it."""
    say("[case] gqa decode, steps in turn", n_keys, nh, nkv, hd)
    c = synth.cfg1_gqa_decode(n_keys, nh, nkv, hd, seed=95)
    cache = hip.KVCache(n_keys, nkv, hd)
    cache.write(0, c["k"], c["v"])
    got = hip.gqa_decode(cache, n_keys, c["q"], c["scale"])
    ref = orc.gqa_decode(c["q"], c["k"], c["v"], c["scale"], nthreads=0)
    # fp32 sums of exact products, as at the other lengths
    assert np.abs(got - ref).max() < 2e-5 * np.abs(ref).max()
    cache.free()


@pytest.mark.parametrize("nh,nkv,hd", [(16, 4, 256), (64, 8, 128), (64, 4, 128)])
def test_gqa_decode_late_maximum_and_dead_lists(hip, orc, nh, nkv, hd):
    """A score far above its wave's first tile (the reference moves), and lists whose first tiles, or
    all of whose entries, name no row."""
    n = 1500
    c = synth.cfg1_gqa_decode(n, nh, nkv, hd, seed=81)
    k = synth.bf16_to_f32(c["k"])
    k[1300] = 25.0 * synth.bf16_to_f32(c["q"]).reshape(nkv, nh // nkv, hd)[:, 0]
    k = synth.f32_to_bf16(k)
    cache = hip.KVCache(n, nkv, hd)
    cache.write(0, k, c["v"])
    got = hip.gqa_decode(cache, n, c["q"], c["scale"])
    ref = orc.gqa_decode(c["q"], k, c["v"], c["scale"], nthreads=0)
    assert np.abs(got - ref).max() < 1e-4 * np.abs(ref).max()
    sel = np.full(700, -1, np.int32)
    sel[400:] = np.arange(300) * 5
    sel[450] = n + 7
    live = sel[(sel >= 0) & (sel < n)]
    got = hip.gqa_decode_sel(cache, sel, c["q"], c["scale"])
    ref = orc.gqa_decode(c["q"], k[live], c["v"][live], c["scale"], nthreads=0)
    assert np.abs(got - ref).max() < 1e-4 * np.abs(ref).max()
    assert (hip.gqa_decode_sel(cache, np.full(100, -1, np.int32), c["q"], c["scale"]) == 0).all()
    cache.free()


@pytest.mark.parametrize("nh,nkv,hd,n_list", [
    (64, 8, 128, 1), (64, 8, 128, 17), (64, 8, 128, 63), (32, 4, 256, 65), (16, 16, 256, 191),    # one workgroup per kv head
    (64, 64, 128, 1089),     # five tiles a wave: one more than the four whose entries it holds at once
    (64, 64, 128, 2049),     # nine
    (128, 64, 128, 3333), (64, 4, 128, 3000),
])
def test_gqa_decode_list_lengths(hip, orc, nh, nkv, hd, n_list):
    """Lists that end inside a tile, a workgroup's step and the four tiles whose entries a wave holds; a fifth of the
    entries name no row, on either side of the range."""
    say("[case] gqa decode, list lengths", nh, nkv, hd, n_list)
    n = 700
    c = synth.cfg1_gqa_decode(n, nh, nkv, hd, seed=92)
    g = synth.rng(93)
    sel = g.integers(0, n, n_list).astype(np.int32)
    bad = g.permutation(n_list)[:n_list // 5]
    sel[bad] = np.where(bad % 2 == 0, -1 - bad, n + bad)
    sel[:n_list:97] = g.integers(0, n, len(sel[:n_list:97]))
    live = sel[(sel >= 0) & (sel < n)]
    cache = hip.KVCache(n, nkv, hd)
    cache.write(0, c["k"], c["v"])
    got = hip.gqa_decode_sel(cache, sel, c["q"], c["scale"])
    ref = orc.gqa_decode(c["q"], c["k"][live], c["v"][live], c["scale"], nthreads=0)
    # fp32 sums of exact products over up to 3333 entries, as in the decode without a list
    assert np.abs(got - ref).max() < 2e-5 * np.abs(ref).max()
    cache.free()


@pytest.mark.parametrize("n,pos0,nh", [
    (1, 5000, 16),           # a quarter of a group, its keys in slices
    (6, 189, 16),            # groups of four queries that end on either side of a tile, nothing to slice
    (5, 3000, 24),           # two row blocks per query, the second half empty; groups of two queries
    (67, 1000, 96),          # six row blocks per query: every other group spans two queries
    (300, 700, 64),          # one full round of whole groups, the rest in slices
    (2, 9000, 128),          # two groups per query, 64 slices
])
def test_mla_prefill_groups_and_slices(hip, orc, n, pos0, nh):
    say("[case] mla prefill groups and slices", n, pos0, nh)
    c = synth.cfg4_mla_prefill(n, pos0, nh, seed=82)
    cache = hip.LatentCache(1, pos0 + n)
    cache.write(0, 0, c["rows"], c["scales"])
    got = hip.mla_prefill_chunk(cache, 0, pos0, c["q"], c["scale"])
    ref = orc.mla_prefill_chunk(c["q"], c["rows"], c["scales"], pos0, c["scale"], nthreads=0)
    assert_close(got, ref, "mla prefill groups", strict=pos0 >= 200)
    cache.free()


@pytest.mark.parametrize("nh", [16, 64])
@pytest.mark.parametrize("n_keys", [191, 192, 193, 256, 257, 320])
def test_mla_prefill_last_tile(hip, orc, n_keys, nh):
    """Lengths around a whole tile: the tiles behind the second are copied from constant lane offsets when they
    are whole, row by row when they are not (the rows past the end then come from a row of zeros)."""
    n = 5
    say("[case] mla prefill last tile", n_keys, nh)
    c = synth.cfg4_mla_prefill(n, n_keys - n, nh, seed=91)
    cache = hip.LatentCache(1, n_keys + 64)
    cache.write(0, 0, c["rows"], c["scales"])
    cache.write(0, n_keys, np.full((64, synth.KDIM), 0x7F, np.uint8), np.full((64, synth.NBLK), np.nan, np.float32))
    got = hip.mla_prefill_chunk(cache, 0, n_keys - n, c["q"], c["scale"])
    ref = orc.mla_prefill_chunk(c["q"], c["rows"], c["scales"], n_keys - n, c["scale"], nthreads=0)
    assert_close(got, ref, "mla prefill, last tile", strict=False)
    cache.free()


@pytest.mark.parametrize("n,pos0,nh", [(8, 20000, 128), (1, 5000, 16), (5, 3000, 24), (300, 700, 64)])
def test_mla_prefill_slices_keep_their_sums(hip, n, pos0, nh):
    """The keys of a group in slices: what the slices hand to the merge has all its bits.  A query of zeros
    weighs every key the same, and rows of small whole numbers with unit scales make every product and
    every sum exact in fp32 (below 2^24), in a slice and over all of them.  What is left is the
    reciprocal of the key count and the multiplication by it: half a unit in the last place each, 2^-23
    together; twice that is allowed.  (Sums handed over in 16 bits are off by 2^-16 of the largest.)"""
    import torch
    say("[case] mla prefill, sums of slices", n, pos0, nh)
    g = synth.rng(88)
    vals = g.integers(-7, 8, (pos0 + n, synth.KDIM)).astype(np.float32)
    rows = torch.from_numpy(vals).to(torch.float8_e4m3fn).view(torch.uint8).numpy()
    cache = hip.LatentCache(1, pos0 + n)
    cache.write(0, 0, rows, np.ones((pos0 + n, synth.NBLK), np.float32))
    got = hip.mla_prefill_chunk(cache, 0, pos0, np.zeros((n, nh, synth.KDIM), np.uint16), 0.1).astype(np.float64)
    sums = np.cumsum(vals[:, :synth.VDIM].astype(np.float64), axis=0)[pos0:]
    ref = (sums / (pos0 + 1 + np.arange(n))[:, None])[:, None, :]
    assert (np.abs(got - ref) <= 2.0 ** -22 * np.abs(ref)).all(), "rel %.2e" % (np.abs(got - ref).max() / np.abs(ref).max())
    cache.free()


@pytest.mark.parametrize("pos0", [61, 64, 700])
def test_mla_prefill_later_rows_stay_out(hip, orc, pos0):
    """Queries that share a workgroup: a later query's row of NaN bytes, or with a scale far above the
    others, changes nothing for the queries before it."""
    n, nh = 4, 16
    say("[case] mla prefill later rows", pos0)
    c = synth.cfg4_mla_prefill(n, pos0, nh, seed=83)
    rows, scales = c["rows"].copy(), c["scales"].copy()
    rows[pos0 + 3] = 0x7F
    scales[pos0 + 2] *= 2.0 ** 12
    cache = hip.LatentCache(1, pos0 + n)
    cache.write(0, 0, rows, scales)
    got = hip.mla_prefill_chunk(cache, 0, pos0, c["q"], c["scale"])
    ref = orc.mla_prefill_chunk(c["q"][:2], rows, scales, pos0, c["scale"], nthreads=0)
    assert_close(got[:2], ref, "mla prefill, later rows", strict=False)
    ref = orc.mla_prefill_chunk(c["q"], rows, scales, pos0, c["scale"], nthreads=0)[2]
    assert np.abs(got[2] - ref).max() <= 1e-2 * np.abs(ref).max()
    assert np.isnan(got[3]).all()
    cache.free()


@pytest.mark.parametrize("ih", [1, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("n_keys", [1, 16, 65, 1000])
def test_indexer_scores_few_keys(hip, orc, n_keys, ih):
    """A key and four heads per lane: bit-equal whatever part of the last workgroup and head group is there."""
    say("[case] indexer scores, few keys", n_keys, ih)
    c = synth.cfg5_dsa(n_keys=n_keys, batch=1, ih=ih, topk=1, nh=16, seed=84)
    ik = hip.IndexKeys(1, n_keys)
    ik.write(0, 0, c["ikeys"][0], c["ikscale"][0])
    got = hip.indexer_scores(ik, 0, n_keys, c["q_idx"][0], c["w"][0])
    ref = orc.indexer_scores(c["q_idx"][0], c["w"][0], c["ikeys"][0], c["ikscale"][0], nthreads=0)
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))
    ik.free()


@pytest.mark.parametrize("n", [1, 1025, 4097, 8192, 8193, 12289, 16385, 24577, 32768, 32769])
@pytest.mark.parametrize("kind", ["smooth", "ties", "equal", "nan"])
def test_topk_register_rows(hip, orc, n, kind):
    """Row lengths on either side of every instantiation; thresholds found after two digits and after
    three, ties that do not all fit, a row of one value, NaNs in the selection."""
    say("[case] topk", n, kind)
    g = synth.rng(85)
    x = g.standard_normal(n, dtype=np.float32)
    if kind == "ties":
        x = np.round(x * 4) / 4
    elif kind == "equal":
        x[:] = -1.5
    elif kind == "nan":
        x[g.permutation(n)[:n // 2 + 1]] = np.nan
    for k in sorted({1, max(1, n // 3), max(1, (2 * n) // 3), n, n + 3}):
        assert np.array_equal(hip.topk(x, k), orc.topk_contract(x, k)), "k %d" % k


@pytest.mark.parametrize("n_keys,batch,topk", [(8192, 8, 512), (8193, 9, 2048), (14337, 4, 700),
                                               (6145, 8, 1000), (65537, 1, 2048), (40003, 2, 512),    # 512 keys a workgroup
                                               (60001, 3, 1024), (65536, 4, 512), (33000, 10, 512),   # 768, 1024, 1536
                                               (33000, 17, 300)])                                     # 2048
def test_dsa_band_of_short_rows(hip, orc, n_keys, batch, topk):
    """The banded select at its shortest rows: four and five stretches of keys per row."""
    say("[case] dsa band, short rows", n_keys, batch, topk)
    c = synth.cfg5_dsa(n_keys=n_keys, batch=batch, ih=64, topk=topk, nh=16, seed=86)
    ik, lat = hip.IndexKeys(batch, n_keys), hip.LatentCache(batch, n_keys)
    for b in range(batch):
        ik.write(b, 0, c["ikeys"][b], c["ikscale"][b])
        lat.write(b, 0, c["rows"][b], c["scales"][b])
    _, sel = hip.dsa_decode(ik, lat, 0, 1, n_keys, c["q_idx"], c["w"], topk, c["q"], c["scale"])
    for b in range(batch):
        sc = orc.indexer_scores(c["q_idx"][b], c["w"][b], c["ikeys"][b], c["ikscale"][b], nthreads=0)
        assert np.array_equal(sel[b], orc.topk_contract(sc, topk)), "query %d" % b
    ik.free()
    lat.free()


@pytest.mark.parametrize("repeats", [2, 7, 60, 400])
def test_dsa_band_ties(hip, orc, repeats):
    """Every key several times over, in places all over the row: the last selected position is one of several with
    the same score, among a candidate list of less and of more than 256."""
    n_keys, batch, topk = 21000, 3, 1024
    say("[case] dsa band, ties", repeats)
    c = synth.cfg5_dsa(n_keys=n_keys, batch=batch, ih=64, topk=topk, nh=16, seed=88)
    ik, lat = hip.IndexKeys(batch, n_keys), hip.LatentCache(batch, n_keys)
    g = np.random.default_rng(3)
    keys, scales = [], []
    for b in range(batch):
        of = g.permutation(n_keys) // repeats
        keys.append(np.ascontiguousarray(c["ikeys"][b][of]))
        scales.append(np.ascontiguousarray(c["ikscale"][b][of]))
        ik.write(b, 0, keys[b], scales[b])
        lat.write(b, 0, c["rows"][b], c["scales"][b])
    _, sel = hip.dsa_decode(ik, lat, 0, 1, n_keys, c["q_idx"], c["w"], topk, c["q"], c["scale"])
    for b in range(batch):
        sc = orc.indexer_scores(c["q_idx"][b], c["w"][b], keys[b], scales[b], nthreads=0)
        assert np.array_equal(sel[b], orc.topk_contract(sc, topk)), "query %d" % b
    ik.free()
    lat.free()


@pytest.mark.parametrize("weights", ["signed", "positive", "equal", "negative"])
@pytest.mark.parametrize("keys", ["independent", "common", "small with empty rows"])
def test_dsa_band_takes_every_kind_of_score(hip, orc, weights, keys):
    """Scores of one sign lie within an octave or two, keys with a common component closer still: the
    threshold's counter has to be narrow enough for the candidate list there as well.  The scratch
    scores tell: a row on the band keeps numbers for its candidates alone, a row that fell back for all
    of its keys.  At 7 bits of fraction the threshold's counter holds 50 to 250 keys of these rows
    (counted on the CPU), and the error bound's band a few dozen more; 12 leading bits held 400 to 5500."""
    import torch
    say("[case] dsa band", weights, keys)
    n_keys, batch, topk, ih = 65536, 2, 2048, 64
    c = synth.cfg5_dsa(n_keys=n_keys, batch=batch, ih=ih, topk=topk, nh=16, shared=False, seed=89)
    g = synth.rng(90)
    w = c["w"]
    w = {"signed": w, "positive": np.abs(w), "equal": np.full_like(w, 0.011), "negative": -np.abs(w)}[weights]
    kb, ks = c["ikeys"], c["ikscale"]
    if keys != "independent":
        x = g.standard_normal((batch, n_keys, 128), dtype=np.float32)
        if keys == "common":
            x += g.standard_normal((batch, 1, 128), dtype=np.float32)
        else:
            x *= np.float32(1e-3)
            x[:, ::3] = 0.0                                   # quantised to zeros with a scale of 1
        amax = np.abs(x).max(axis=2)
        ks = np.where(amax > 0, amax / 448.0, 1.0).astype(np.float32)
        kb = torch.from_numpy(np.clip(x / ks[:, :, None], -448, 448)).to(torch.float8_e4m3fn).view(torch.uint8).numpy()
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    ops = [d(kb), d(ks), d(c["rows"]), d(c["scales"]), d(c["q_idx"].view(np.int16)), d(w), d(c["q"].view(np.int16))]
    tmp = torch.empty((batch, n_keys), dtype=torch.float32, device="cuda")
    sel = torch.empty((batch, topk), dtype=torch.int32, device="cuda")
    out = torch.empty((batch, 16, synth.VDIM), dtype=torch.float32, device="cuda")
    hip.dsa_decode_dev(ops[0], ops[1], n_keys * 128, n_keys, ops[2], ops[3], n_keys * synth.KDIM, n_keys * synth.NBLK, batch,
                       n_keys, ops[4], ops[5], ih, topk, ops[6], 16, c["scale"], tmp, sel, out,
                       torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    kept = torch.isfinite(tmp).sum(dim=1).tolist()
    say("[band] candidates", kept)
    for b in range(batch):
        sc = orc.indexer_scores(c["q_idx"][b], w[b], kb[b], ks[b], nthreads=0)
        assert np.array_equal(sel[b].cpu().numpy(), orc.topk_contract(sc, topk)), "query %d" % b
        # (negative weights and empty rows: 20000 keys tie for the best score, 0, whatever the counters)
        ties = weights == "negative" and keys == "small with empty rows"
        assert kept[b] <= 512 or ties, "query %d: %d candidates" % (b, kept[b])


@pytest.mark.parametrize("limit,ih,block,keep", [(1, 1, 64, 1), (63, 3, 64, 2), (130, 5, 128, 4), (1000, 2, 100, 3), (66000, 8, 64, 16),
                                                 (70000, 4, 17, 8)])
def test_mm_select_edges(hip, orc, limit, ih, block, keep):
    """Head counts between the instantiations, one position, rows of more than 1024 and of more than 4096 blocks,
    and blocks that are no whole number of groups."""
    import torch
    say("[case] mm select edges", limit, ih, block, keep)
    g = synth.rng(87)
    keys = synth.f32_to_bf16(g.standard_normal((limit, 128), dtype=np.float32))
    iq = g.standard_normal((1, ih, 128), dtype=np.float32)
    s = torch.cuda.current_stream().cuda_stream
    d_k, d_q = torch.from_numpy(keys.view(np.int16)).cuda(), torch.from_numpy(iq).cuda()
    scores = torch.empty((1, limit), dtype=torch.float32, device="cuda")
    max_sel = (keep + 1) * block
    sel = torch.empty((1, max_sel), dtype=torch.int32, device="cuda")
    hip.mm_select_dev(d_k, d_q, 1, limit, ih, 128, block, keep, scores, limit, None, sel, max_sel, None, s)
    torch.cuda.synchronize()
    ref = orc.mm_index_scores(iq[0], keys, limit)
    got = scores[0].cpu().numpy()
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), "scores are one chain per head in dimension order"
    best = orc.topk_contract(np.array([max(ref[b:b + block].max(), -1e30) for b in range(0, limit, block)], np.float32), keep)
    blocks = sorted({int(b) for b in best if b >= 0} | {limit // block})
    want = [p for b in blocks for p in range(b * block, min(limit, (b + 1) * block))]
    have = sel[0].cpu().numpy()
    assert have[have >= 0].tolist() == want[:max_sel]


@pytest.mark.parametrize("limit,block,keep,kind", [
    (1, 64, 16, "random"), (4095, 64, 64, "random"), (4096, 64, 64, "random"), (4097, 64, 65, "random"),     # 64 blocks, 64 and 65 kept
    (32766, 64, 8, "few levels"), (32767, 64, 8, "few levels"),             # 512 and 513 blocks of the last query: one, four a thread
    (32768, 64, 8, "few levels"), (32769, 64, 8, "few levels"),
    (82000, 64, 16, "random"), (110000, 64, 33, "few levels"),              # live blocks in the later waves
    (131070, 64, 16, "random"), (131071, 64, 16, "random"),                 # 2048 blocks of the last query, and one too many
    (131070, 64, 16, "equal"), (131070, 64, 32, "few levels"), (131070, 64, 64, "ascending"), (131070, 64, 64, "few levels"),
    (131072, 64, 16, "random"), (131073, 64, 16, "random"),
    (65536, 256, 16, "ascending"), (65500, 128, 16, "equal"), (9000, 64, 64, "few levels"), (9000, 128, 3, "negative")])
def test_mm_pick_of_few_blocks(hip, orc, limit, block, keep, kind):
    """A selection of up to 64 of up to 2048 blocks: as many blocks as lanes, candidates for the threshold that fit a wave's
    lanes and that do not, ties that do not all fit, and the line to the radix select of longer rows; three queries
    of growing limits (the last one's blocks pick the kernel).  The scores are set by one dimension, so that whole blocks agree."""
    import torch
    say("[case] mm pick", limit, block, keep, kind)
    g = synth.rng(91)
    n, nq = limit + 2, 3
    nb = (n + block - 1) // block
    level = {"random": g.standard_normal(nb), "few levels": g.integers(0, 4, nb) - 1.0, "ascending": np.arange(nb) / 64.0 + 1.0,
             "equal": np.ones(nb), "negative": -np.ones(nb)}[kind]
    keys = np.zeros((n, 128), np.float32)
    keys[:, 5] = level.repeat(block)[:n]
    keys = synth.f32_to_bf16(keys)
    iq = np.ones((nq, 1, 128), np.float32)
    d_k, d_q = torch.from_numpy(keys.view(np.int16)).cuda(), torch.from_numpy(iq).cuda()
    scores = torch.empty((nq, n), dtype=torch.float32, device="cuda")
    max_sel = (keep + 1) * block
    sel = torch.empty((nq, max_sel), dtype=torch.int32, device="cuda")
    blk = torch.empty((nq, keep + 1), dtype=torch.int32, device="cuda")
    n_sel = torch.empty(nq, dtype=torch.int32, device="cuda")
    hip.mm_select_dev(d_k, d_q, nq, limit, 1, 128, block, keep, scores, n, blk, sel, max_sel, n_sel,
                      torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    for y in range(nq):
        lim = limit + y
        ref = orc.mm_index_scores(iq[y], keys, lim)
        assert np.array_equal(scores[y, :lim].cpu().numpy(), ref)
        best = orc.topk_contract(np.array([max(ref[b:b + block].max(), -1e30) for b in range(0, lim, block)], np.float32), keep)
        blocks = sorted({int(b) for b in best if b >= 0} | {lim // block})
        assert [b for b in blk[y].tolist() if b >= 0] == blocks, "query %d" % y
        want = [p for b in blocks for p in range(b * block, min(lim, (b + 1) * block))][:max_sel]
        have = sel[y].cpu().numpy()
        assert have[have >= 0].tolist() == want and int(n_sel[y]) == len(want), "query %d" % y


def _mm_pick(hip, torch, level, limit, block, keep):
    """A selection over keys whose scores are `level`, one value a block; as a call to repeat, and its list of blocks."""
    keys = np.zeros((limit, 128), np.float32)
    keys[:, 5] = np.asarray(level, np.float32).repeat(block)[:limit]
    keys = synth.f32_to_bf16(keys)
    d_k, d_q = torch.from_numpy(keys.view(np.int16)).cuda(), torch.ones((1, 1, 128), device="cuda")
    scores = torch.empty((1, limit), dtype=torch.float32, device="cuda")
    sel = torch.empty((1, (keep + 1) * block), dtype=torch.int32, device="cuda")
    blk = torch.empty((1, keep + 1), dtype=torch.int32, device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    call = lambda: hip.mm_select_dev(d_k, d_q, 1, limit, 1, 128, block, keep, scores, limit, blk, sel, (keep + 1) * block,
                                     None, s)
    return keys, call, blk, sel


@pytest.mark.parametrize("limit,block,keep,kind", [
    (131072, 64, 32, "random"), (131072, 64, 33, "random"), (65536, 128, 64, "random"),     # the line to the radix select
    (131072, 64, 32, "same lanes"), (65536, 64, 32, "same lanes"),          # three bits a turn down to the last ones
    (32768, 64, 32, "same lanes"), (131072, 64, 32, "next to one another"), (32768, 64, 31, "next to one another"),
    (131072, 64, 16, "equal"), (32768, 64, 16, "zero"), (131072, 64, 1, "equal"), (4161, 64, 32, "equal"),
    (131072, 64, 16, "100 top"), (32768, 64, 16, "100 top"),                # ties above all others, spread over the waves
    (131072, 64, 32, "20 above 100"), (32768, 64, 32, "20 above 100"),      # some above the ties, twelve of the ties
    (131072, 64, 16, "late")])                                              # ties in the last wave only
def test_mm_pick_of_many_candidates(hip, orc, limit, block, keep, kind):
    """A selection in which more than 64 blocks reach its bound, by counts of the whole workgroup, and the line to
    the radix select."""
    import torch
    say("[case] mm pick, many candidates", limit, block, keep, kind)
    g = synth.rng(92)
    nb = (limit + block - 1) // block
    level = np.ones(nb)
    some = g.permutation(nb)
    if kind == "random":
        level = 1.0 + np.abs(g.standard_normal(nb))
    elif kind == "zero":
        level = np.zeros(nb)
    elif kind == "100 top":
        level[some[:100]] = 2.0
    elif kind == "20 above 100":
        level[some[:20]], level[some[20:120]] = 3.0 + g.integers(0, 3, 20), 2.0
    elif kind == "same lanes": # the best in one lane of every wave
        level = 1.0 + 0.5 * g.random(nb)
        level[17::64] = 2.0 ** g.integers(1, 20, len(level[17::64])) * (1.0 + 0.9 * g.random(len(level[17::64])))
    elif kind == "next to one another":
        level = 1.0 + g.integers(0, 128, nb) / 128.0                        # neighbours in bf16
    elif kind == "late":
        level[-100:] = 2.0
    keys, call, blk, sel = _mm_pick(hip, torch, level, limit, block, keep)
    call()
    torch.cuda.synchronize()
    ref = orc.mm_index_scores(np.ones((1, 128), np.float32), keys, limit)
    best = orc.topk_contract(np.array([ref[b:b + block].max() for b in range(0, limit, block)], np.float32), keep)
    blocks = sorted({int(b) for b in best if b >= 0} | {limit // block})
    assert [b for b in blk[0].tolist() if b >= 0] == blocks
    want = [p for b in blocks for p in range(b * block, min(limit, (b + 1) * block))]
    have = sel[0].cpu().numpy()
    assert have[have >= 0].tolist() == want


@pytest.mark.parametrize("keep,kind", [(16, "equal"), (64, "random")])
def test_mm_pick_of_many_candidates_is_no_slow_path(hip, keep, kind):
    """2048 blocks that all tie, and 64 kept of 2048, in less than 2.5 times what sixteen of distinct ones take (1.0 and 1.3
    times; by counts of one wave alone 5.8 and 4)."""
    import torch
    say("[case] mm pick, time of many candidates", keep, kind)

    def us(level, keep):
        _, call, _, _ = _mm_pick(hip, torch, level, 131072, 64, keep)
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        best = []
        for _ in range(7):
            a.record()
            for _ in range(100):
                call()
            b.record()
            torch.cuda.synchronize()
            best.append(a.elapsed_time(b) * 10.0)
        return min(best)
    distinct = np.random.default_rng(93).permutation(2048) / 2048.0 + 1.0
    base, many = us(distinct, 16), us(np.ones(2048) if kind == "equal" else distinct, keep)
    say("[time]", base, many)
    assert many < 2.5 * base


@pytest.mark.parametrize("splits", [1, 2, 4, 5, 8, 9, 16, 17, 31, 32, 33, 64, 65, 127, 128, 129, 200, 255])
def test_merges_of_every_number_of_slices(hip, orc, splits):
    """As many 64-key slices as the merge of a GQA decode (one kv head) takes at a time, one more and one fewer, the last
    slice a single key, one slice far above the others; and an MLA decode (16 heads) over as many keys, which
    it cuts into fewer slices from 108 tiles on (their numbers: MLA_SLICES)."""
    say("[case] merges", splits)
    n = 64 * (splits - 1) + 1
    c = synth.cfg1_gqa_decode(n_keys=n, nh=8, nkv=1, hd=128, seed=splits)
    top = synth.bf16_to_f32(c["q"][3]) * np.float32(3.0)          # a key that one head agrees with
    c["k"][n // 2, 0] = synth.f32_to_bf16(top)
    kv = hip.KVCache(n, 1, 128)
    kv.write(0, c["k"].reshape(n, -1), c["v"].reshape(n, -1))
    got = hip.gqa_decode(kv, n, c["q"], c["scale"])
    ref = orc.gqa_decode(c["q"], c["k"], c["v"], c["scale"], nthreads=0)
    assert np.isfinite(got).all() and np.abs(got - ref).max() <= 2e-3
    c = synth.cfg3_mla_decode(n, 16, seed=splits)
    lat = hip.LatentCache(1, n)
    lat.write(0, 0, c["rows"], c["scales"])
    got = hip.mla_decode(lat, 0, c["q"], c["scale"], n_list=n)
    ref = orc.mla_decode(c["q"], c["rows"], c["scales"], c["scale"], nthreads=0)
    assert np.isfinite(got).all() and (np.abs(got - ref) <= 2e-3 + 1e-2 * np.abs(ref)).all()


# Keys, heads and queries of an MLA decode, and the slices that they are cut into with 256 compute units
# (test_host_rules.py has the rule give these numbers).  Where there is one query, the last slice is a single key.
MLA_SLICES = [
    (193, 32, 64, 2), (385, 16, 1, 7), (449, 16, 1, 8), (513, 16, 1, 9),        # up to eight: a wave by itself
    (2049, 16, 1, 33), (4033, 16, 1, 64), (4097, 16, 1, 65),                    # four of eight waves each, eight, sixteen waves
    (16129, 16, 1, 127), (16257, 16, 1, 128), (16385, 16, 1, 129),              # eight of sixteen waves each, and one more
    (17281, 16, 1, 136), (18433, 32, 1, 97), (30529, 16, 1, 160), (49153, 16, 1, 193), (65281, 32, 1, 256),
]


@pytest.mark.parametrize("n,nh,batch,slices", MLA_SLICES)
def test_mla_merge_of_every_number_of_slices(hip, orc, n, nh, batch, slices):
    """The merge of an MLA decode: as many slices as it takes at a time, one more and one fewer, up to a full round of
    them; a key in the middle whose slice has the greatest maximum by far."""
    import torch
    say("[case] mla merge", n, nh, batch, slices)
    c = synth.cfg3_mla_decode(n, nh, seed=n + nh)
    c["scales"][n // 2] *= np.float32(6.0)
    g = synth.rng(n)
    q = synth.f32_to_bf16(g.standard_normal((batch, nh, synth.KDIM), dtype=np.float32))
    d_rows, d_scales = torch.from_numpy(c["rows"]).cuda(), torch.from_numpy(c["scales"]).cuda()
    out = torch.full((batch, nh, synth.VDIM), float("nan"), device="cuda")
    # (a stride of 0: the queries share the rows)
    hip.mla_decode_dev(d_rows, d_scales, 0, 0, n, batch, None, n, torch.from_numpy(q.view(np.int16)).cuda(), nh, c["scale"],
                       out, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    for y in {0, batch // 2, batch - 1}:
        ref = orc.mla_decode(q[y], c["rows"], c["scales"], c["scale"], nthreads=0)
        got = out[y].cpu().numpy()
        assert np.isfinite(got).all() and (np.abs(got - ref) <= 2e-3 * np.abs(ref).max() + 1e-2 * np.abs(ref)).all()


@pytest.mark.parametrize("n_keys,ih,kind", [(31, 32, "normal"), (513, 33, "normal"), (4111, 1, "normal"),
                                            (777, 32, "one dim"), (777, 64, "tiny"), (777, 32, "huge"),
                                            (600, 32, "infinite"), (600, 64, "nan key")])
def test_indexer_bound_row(hip, orc, n_keys, ih, kind):
    """The bound of the approximate scores where its E4M3 coefficients have an edge: one or two blocks of
    heads, a coefficient far above the others, magnitudes near the ends of fp32, an infinite query, a NaN key."""
    import torch
    say("[case] indexer bound row", n_keys, ih, kind)
    g = synth.rng(640 + n_keys + ih)
    keys, ks = synth.index_keys(g, n_keys)
    q = synth.normal_bf16(g, (ih, synth.IDIM))
    w = (g.standard_normal(ih, dtype=np.float32) / np.float32(np.sqrt(128.0 * ih))).astype(np.float32)
    if kind == "one dim":
        qf = synth.bf16_to_f32(q)
        qf[:, 77] *= np.float32(2.0 ** 20)
        q = synth.f32_to_bf16(qf)
    elif kind in ("tiny", "huge"):
        w = (w * np.float32(2.0 ** (-100 if kind == "tiny" else 100))).astype(np.float32)
    elif kind == "infinite":
        q = q.copy()
        q[ih - 1, 5] = 0x7F80
    elif kind == "nan key":
        keys = keys.copy()
        keys.reshape(n_keys, 128)[n_keys - 1, 100] = 0x7F
    cache = hip.IndexKeys(1, n_keys)
    cache.write(0, 0, keys, ks)
    approx, bound = hip.indexer_scores_approx(cache, 0, n_keys, q, w)
    if kind in ("infinite", "nan key"):
        assert not np.isfinite(bound)                       # the row is scored exactly
        return
    ref = orc.indexer_scores(q, w, keys, ks, nthreads=0)
    # the bound in 64 bits; a coefficient is rounded up by an eighth at most, one below 2^-13 of the largest to that
    e = np.abs(torch.from_numpy(keys.reshape(n_keys, 128).copy()).view(torch.float8_e4m3fn).double().numpy())
    c = (np.abs(w.astype(np.float64))[:, None] * np.abs(synth.bf16_to_f32(q).astype(np.float64))).sum(axis=0)
    least = ((e @ c) * np.abs(ks.astype(np.float64))).max() * 512.0 / 2 ** 24
    most = ((e @ np.maximum(c * 1.125, c.max() / 2 ** 12)) * np.abs(ks.astype(np.float64))).max() * 512.0 / 2 ** 24
    assert least * (1 - 1e-4) <= bound <= most * (1 + 1e-4)
    assert np.abs(approx.astype(np.float64) - ref.astype(np.float64)).max() <= bound


@pytest.mark.parametrize("n_keys,ih,kind", [(1111, 32, "normal"), (2049, 64, "normal"), (300, 7, "one dim"), (333, 64, "one dim off"),
                                            (500, 33, "subnormal keys"), (97, 16, "halves"), (97, 40, "nothing")])
def test_indexer_bound_has_twelve_bits(hip, orc, n_keys, ih, kind):
    """The bound of the approximate scores against its coefficients in 64 bits: rounded up by a 2048th of their own or by
    2^-21 of the largest at most, less than a coefficient in bf16 is."""
    import torch
    say("[case] indexer bound, twelve bits", n_keys, ih, kind)
    g = synth.rng(660 + n_keys + ih)
    keys, ks = synth.index_keys(g, n_keys)
    qf = synth.bf16_to_f32(synth.normal_bf16(g, (ih, synth.IDIM)))
    w = (g.standard_normal(ih, dtype=np.float32) / np.float32(np.sqrt(128.0 * ih))).astype(np.float32)
    if kind.startswith("one dim"):
        qf[:, 77] *= np.float32(2.0 ** 12)
        if kind == "one dim off":                           # only the other coefficients, and their terms, count
            keys.reshape(n_keys, 128)[:, 77] = 0
    elif kind == "subnormal keys":
        keys = (g.integers(0, 8, (n_keys, 128)) | g.integers(0, 2, (n_keys, 128)) << 7).astype(np.uint8)
    elif kind == "halves":                                  # c = 1/2, 1/4 .. 2^-12: each exact in one term
        qf[:] = 2.0 ** -(1.0 + np.arange(128) % 12) / ih
        w[:] = 1.0
    elif kind == "nothing":
        w[:] = 0.0
    q = synth.f32_to_bf16(qf.astype(np.float32))
    cache = hip.IndexKeys(1, n_keys)
    cache.write(0, 0, keys, ks)
    approx, bound = hip.indexer_scores_approx(cache, 0, n_keys, q, w)
    ref = orc.indexer_scores(q, w, keys, ks, nthreads=0)
    e = np.abs(torch.from_numpy(np.ascontiguousarray(keys).reshape(n_keys, 128).copy()).view(torch.float8_e4m3fn).double().numpy())
    c = (np.abs(w.astype(np.float64))[:, None] * np.abs(synth.bf16_to_f32(q).astype(np.float64))).sum(axis=0)
    unit = np.abs(ks.astype(np.float64)) * 512.0 / 2 ** 24
    least = ((e @ c) * unit).max()
    most = ((e @ (c * (1 + 2.0 ** -11) + (c > 0) * c.max() * 2.0 ** -21)) * unit).max()
    say("[bound]", bound, least, most)
    # Below: of eight products that the FP8 matrix core adds up at a time, each loses its bits under 2^-13 of the largest,
    # so that a sum of products of one sign may lack 7 x 2^-13 of itself (no more than 1.3e-4 was seen over coefficients
    # of twelve octaves).  1e-5: fp32 sums of 3 x 128 terms, and of up to 64 heads in a coefficient.
    assert least * (1 - 7 * 2.0 ** -13 - 1e-5) <= bound <= most * (1 + 1e-5)
    assert np.abs(approx.astype(np.float64) - ref.astype(np.float64)).max() <= bound


@pytest.mark.parametrize("n,nh", [
    (128, 16), (129, 16),            # two tiles in one workgroup, three in three
    (8192, 16),                      # two tiles each instead of one
    (4097, 128), (12288, 128),       # a last workgroup of one tile; four tiles each instead of three
])
def test_mla_decode_fewer_workgroups(hip, orc, n, nh):
    """The lengths at which a workgroup of the MLA decode takes more tiles than a full round of workgroups needs."""
    say("[case] mla decode, fewer workgroups", n, nh)
    c = synth.cfg3_mla_decode(n, nh, seed=n)
    lat = hip.LatentCache(1, n)
    lat.write(0, 0, c["rows"], c["scales"])
    got = hip.mla_decode(lat, 0, c["q"], c["scale"], n_list=n)
    ref = orc.mla_decode(c["q"], c["rows"], c["scales"], c["scale"], nthreads=0)
    assert_close(got, ref, "mla decode, fewer workgroups", strict=False)
    lat.free()


@pytest.mark.parametrize("n_keys", [64, 65, 128, 129, 192, 193, 256, 257, 320, 383])
@pytest.mark.parametrize("listed", [False, True])
def test_mla_decode_tiles_of_a_workgroup(hip, orc, n_keys, listed):
    """One to six tiles in a workgroup, the last one whole and not (256 blocks of 32 heads leave one workgroup to each): the
    steps that copy a whole tile, the ones that copy what there is, and those behind the last copy."""
    import torch
    say("[case] mla decode, tiles of a workgroup", n_keys, listed)
    batch, nh, n_rows = 64, 128, 400
    c = synth.cfg3_mla_decode(n_rows, nh, seed=96)
    g = synth.rng(97)
    q = synth.f32_to_bf16(g.standard_normal((batch, nh, synth.KDIM), dtype=np.float32))
    q[0] = c["q"]
    sel = np.stack([g.permutation(n_rows)[:n_keys] for _ in range(batch)]).astype(np.int32)
    sel[:, n_keys // 3] = -1
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    rows, scales, dq, dsel = d(c["rows"].view(np.uint8)), d(c["scales"]), d(q.view(np.int16)), d(sel)
    out = torch.zeros((batch, nh, synth.VDIM), dtype=torch.float32, device="cuda")
    hip.mla_decode_dev(rows, scales, 0, 0, n_rows, batch, dsel if listed else None, n_keys, dq, nh, c["scale"], out,
                       torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    for y in (0, batch - 1):
        if listed:
            ref = orc.mla_decode(q[y], c["rows"], c["scales"], c["scale"], sel=sel[y], nthreads=0)
        else:
            ref = orc.mla_decode(q[y], c["rows"][:n_keys], c["scales"][:n_keys], c["scale"], nthreads=0)
        assert_close(out[y].cpu().numpy(), ref, "mla decode, tiles of a workgroup", strict=False)


# chunks that 64-row workgroups take, and the steps of four tiles those have, with one-term and with two-term weights (up to
# six and three of them are rounds; tests/test_host_rules.py holds the plan to these figures)
PREFILL_ROUNDS = [
    ((656, 0, 16, 4), (), range(1, 4)),              # slices, the last ones of one to three tiles
    ((645, 0, 8, 8), (), (1, 2)),
    ((1025, 0, 16, 4), (9,), range(1, 9)),           # whole blocks: three rounds with two-term weights, and the other body from four steps on
    ((1300, 200, 8, 8), (9, 10, 11, 12), range(3, 9)),      # diagonals that begin in one round and end in the next
    ((100, 7000, 16, 4), (6, 7), ()),                # slices of six rounds, and of seven steps of the other body
    ((90, 6000, 16, 4), (2, 3, 5), ()),              # slices of five rounds
    ((200, 7000, 16, 4), (10, 11, 12, 15), ()),
    ((9, 8191, 16, 2), (1, 2), ()),                  # slices, the last one of a tile
    ((5, 508, 4, 2), (), (1, 2)),                    # rows of one block only
]


@pytest.mark.parametrize("n,pos0,nh,nkv", [shape for shape, _, _ in PREFILL_ROUNDS])
@pytest.mark.parametrize("late", [0, 1, 4])
def test_gqa_prefill_rounds(hip, orc, n, pos0, nh, nkv, late):
    """Workgroups whose waves pass their weights round, at the number of rounds up to which they do; with keys that outgrow
    every reference before them in several rounds, so that the workgroup starts over."""
    say("[case] gqa prefill, rounds", n, pos0, nh, nkv, late)
    c = synth.cfg2_gqa_prefill(n, nh, nkv, 256, pos0, seed=98)
    k = synth.bf16_to_f32(c["k"])
    for i in range(late):
        k[(pos0 + n) * (i + 1) // (late + 1)] = 20.0 * (i + 1) * synth.bf16_to_f32(c["q"])[n - 1].reshape(nkv, nh // nkv, 256)[:, 0]
    k = synth.f32_to_bf16(k)
    cache = hip.KVCache(pos0 + n, nkv, 256)
    cache.write(0, k.reshape(pos0 + n, -1), c["v"].reshape(pos0 + n, -1))
    got = hip.gqa_prefill(cache, pos0, c["q"], c["scale"])
    ref = orc.gqa_prefill(c["q"], k, c["v"], pos0, c["scale"], nthreads=0)
    assert_close(got, ref, "gqa prefill, rounds", strict=False)
    cache.free()


@pytest.mark.parametrize("listed", [False, True])
@pytest.mark.parametrize("n_keys,nh", [(64, 16), (300, 40), (9000, 64)])
def test_mla_decode_score_that_overflows_when_scaled(hip, orc, n_keys, nh, listed):
    """A score that fp32 holds and whose scaled value it does not: the head's row is NaN, as it is with a score that overflows
    by itself (infinity minus infinity), whether its keys are one slice or several; the other heads' rows are what they are."""
    say("[case] mla decode, overflow when scaled", n_keys, nh, listed)
    c = synth.cfg3_mla_decode(n_keys, nh, seed=99)
    scale, dim, key, head = 3.0, 520, 2 * n_keys // 3, 1          # (a rope dim: no part of any value)
    q, rows, scales = synth.bf16_to_f32(c["q"]) * (c["scale"] / scale), c["rows"].copy(), c["scales"].copy()
    q[:, dim] = 0.0
    q[head, dim] = 5e17
    rows[key, 512:], scales[key, 4] = 0, 1e18
    rows[key, dim] = 0x78                                           # 256: the score is 1.28e38, three times that no fp32 value
    q = synth.f32_to_bf16(q)
    sel = synth.rng(100).permutation(n_keys).astype(np.int32) if listed else None
    lat = hip.LatentCache(1, n_keys)
    lat.write(0, 0, rows, scales)
    got = hip.mla_decode(lat, 0, q, scale, sel=sel, n_list=n_keys)
    ref = orc.mla_decode(q, rows, scales, scale, sel=sel, nthreads=0)
    others = np.arange(nh) != head
    assert np.isnan(ref[head]).all() and np.isnan(got[head]).all()
    assert_close(got[others], ref[others], "mla decode, the other heads", strict=False)
    lat.free()


@pytest.mark.parametrize("n,pos0,nh,nkv", [
    (16, 0, 16, 4),          # one tile
    (100, 0, 16, 4),         # few steps, whole blocks
    (9, 8191, 16, 2),        # few steps, slices
    (1025, 0, 16, 4),        # more steps, whole blocks
    (300, 5000, 16, 4),      # more steps, slices
    (517, 7083, 16, 4),      # 256 rows, slices
    (2000, 0, 32, 4),        # 256 rows, whole blocks
])
@pytest.mark.parametrize("early", [False, True])
def test_gqa_prefill_score_that_overflows_when_scaled(hip, orc, n, pos0, nh, nkv, early):
    """A score that fp32 holds and whose scaled value it does not: the row is NaN, as it is with a score that overflows by
    itself (infinity minus infinity), whichever workgroup it falls to; the other rows are what they are."""
    say("[case] gqa prefill, overflow when scaled", n, pos0, nh, nkv, early)
    c = synth.cfg2_gqa_prefill(n, nh, nkv, 256, pos0, seed=101)
    scale, dim, key, head, row = 3.0, 17, 3 if early else 2 * (pos0 + n) // 3, 1, n - 1
    q, k = synth.bf16_to_f32(c["q"]) * (c["scale"] / scale), synth.bf16_to_f32(c["k"])
    q[:, :, dim] = 0.0
    q[row, head, dim] = k[key, head // (nh // nkv), dim] = 1.2e19           # the score is 1.4e38, three times that no fp32 value
    q, k = synth.f32_to_bf16(q), synth.f32_to_bf16(k)
    cache = hip.KVCache(pos0 + n, nkv, 256)
    cache.write(0, k.reshape(pos0 + n, -1), c["v"].reshape(pos0 + n, -1))
    got = hip.gqa_prefill(cache, pos0, q, scale)
    ref = orc.gqa_prefill(q, k, c["v"], pos0, scale, nthreads=0)
    assert np.isnan(ref[row, head]).all() and np.isnan(got[row, head]).all()
    others = ~((np.arange(n) == row)[:, None] & (np.arange(nh) == head))
    assert_close(got[others], ref[others], "gqa prefill, the other rows", strict=False)
    cache.free()
