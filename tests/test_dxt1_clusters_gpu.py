"""Wave-per-cluster DXT1 search (dxt_hc endpoint clusters of 1 to thousands of
texels) against the oracle's optimizer on the same texels: error and
endpoints per cluster, selectors per texel, and the reported error recomputed
from the emitted endpoints and selectors."""
import numpy as np
import pytest
import torch

import oracle
from crunch2_amd import dxt1, texture

pytestmark = pytest.mark.gpu
W = np.array([8, 25, 1], np.int64)


def clusters(seed, sizes):
    rng = np.random.default_rng(seed)
    img = texture.synth(512, 512, seed, texture.RGB).reshape(-1, 4)
    parts = []
    for n in sizes:
        start = int(rng.integers(0, img.shape[0] - n))
        if rng.random() < 0.5:
            parts.append(img[start:start + n])                                   # smooth run of texels
        else:
            parts.append(img[rng.integers(0, img.shape[0], n)])                   # scattered texels
    return parts


@pytest.mark.parametrize("perceptual", [True, False])
def test_clusters_match_oracle(gpu, perceptual):
    rng = np.random.default_rng(5)
    sizes = [1, 2, 3, 4, 16, 17, 64, 200] + list(rng.integers(16, 2048, 40)) + [4096, 5000]
    parts = clusters(6 + perceptual, sizes)
    parts.append(np.repeat(parts[0][:1], 300, axis=0))                            # one colour, many texels
    px = np.concatenate(parts)
    ofs = np.concatenate([[0], np.cumsum([len(p) for p in parts])]).astype(np.int32)
    print("clusters", len(parts), "texels", len(px), flush=True)
    raw, sel = dxt1.encode_clusters_device(torch.from_numpy(px).cuda(), torch.from_numpy(ofs).cuda(), perceptual)
    torch.cuda.synchronize()
    r = raw.cpu().numpy().view(dxt1.CLUSTER_DTYPE).reshape(-1)
    sel = sel.cpu().numpy()
    flags = oracle.DXT1_PERCEPTUAL if perceptual else 0
    same, same_err = 0, 0
    for c, p in enumerate(parts):
        osel, ores = oracle.dxt1_cluster(p, 4, flags)
        lo, hi = int(r["lo_hi"][c] & 0xFFFF), int(r["lo_hi"][c] >> 16)
        s = sel[ofs[c]:ofs[c + 1]]
        e = int(r["error"][c])
        same_err += e == ores.error
        same += e == ores.error and lo == ores.low and hi == ores.high and np.array_equal(s, osel)
        # the reported error is the emitted block's (hc palette with the alternate-rounding flag)
        alt = int((r["flags"][c] >> 2) & 1)

        def ex(v):
            return np.array([((v >> 11) & 31) * 33 // 4, ((v >> 5) & 63) * 65 // 16, (v & 31) * 33 // 4], np.int64)
        c0, c1 = ex(lo), ex(hi)
        pal = np.stack([c0, c1, (2 * c0 + c1 + alt) // 3, (c0 + 2 * c1 + alt) // 3])
        d = ((p[:, None, :3].astype(np.int64) - pal[None]) ** 2 * (W if perceptual else 1)).sum(-1)
        if not (r["flags"][c] >> 3) & 1:
            assert int(d[np.arange(len(p)), s].sum()) == e, c
    print("bit-exact clusters %d / %d, error-equal %d" % (same, len(parts), same_err), flush=True)
    assert same_err >= len(parts) - 1
    assert same >= len(parts) - 2


@pytest.mark.parametrize("perceptual", [True, False])
def test_clusters_beyond_the_lds_store(gpu, perceptual):
    # clusters of more than 4,096 distinct colours take the global-memory pass
    rng = np.random.default_rng(11)
    img = texture.synth(512, 512, 30 + perceptual, texture.RGB).reshape(-1, 4)
    noisy = rng.integers(0, 256, (9000, 4), dtype=np.uint8)
    parts = [img[:6000], noisy, img[rng.integers(0, img.shape[0], 20000)], img[100:164], noisy[:3000]]
    px = np.concatenate(parts)
    ofs = np.concatenate([[0], np.cumsum([len(p) for p in parts])]).astype(np.int32)
    print("big clusters", [len(p) for p in parts], [len(np.unique(p[:, :3].view(np.uint8).reshape(-1, 3), axis=0))
                                                  for p in parts], flush=True)
    raw, sel = dxt1.encode_clusters_device(torch.from_numpy(px).cuda(), torch.from_numpy(ofs).cuda(), perceptual)
    torch.cuda.synchronize()
    r = raw.cpu().numpy().view(dxt1.CLUSTER_DTYPE).reshape(-1)
    sel = sel.cpu().numpy()
    flags = oracle.DXT1_PERCEPTUAL if perceptual else 0
    for c, p in enumerate(parts):
        assert not (r["flags"][c] >> 8) & 1, c
        osel, ores = oracle.dxt1_cluster(p, 4, flags)
        assert r["nunique"][c] == len(np.unique(p[:, :3], axis=0)), c
        assert int(r["error"][c]) == ores.error, c
        assert (int(r["lo_hi"][c] & 0xFFFF), int(r["lo_hi"][c] >> 16)) == (ores.low, ores.high), c
        assert np.array_equal(sel[ofs[c]:ofs[c + 1]], osel), c


@pytest.mark.parametrize("perceptual", [True, False])
def test_clusters_with_three_colour_blocks_match_oracle(gpu, perceptual):
    # qdxt1's endpoint clusters: the uber evaluator with both block types
    # (crn_dxt1.cpp:1370-1592), solid tries and return_solution with their
    # 3-colour branches; every size class and the global-memory pass
    rng = np.random.default_rng(21)
    sizes = [1, 2, 3, 16, 17, 64, 200] + list(rng.integers(16, 2048, 30)) + [4096, 5000]
    parts = clusters(40 + perceptual, sizes)
    parts.append(np.repeat(parts[0][:1], 300, axis=0))
    parts.append(rng.integers(0, 256, (6000, 4), dtype=np.uint8))
    two = np.zeros((64, 4), np.uint8)
    two[:32, :3], two[32:, :3] = (10, 200, 30), (200, 20, 240)
    parts.append(two)
    px = np.concatenate(parts)
    ofs = np.concatenate([[0], np.cumsum([len(p) for p in parts])]).astype(np.int32)
    print("clusters", len(parts), "texels", len(px), flush=True)
    raw, sel = dxt1.encode_clusters_device(torch.from_numpy(px).cuda(), torch.from_numpy(ofs).cuda(), perceptual,
                                           alpha_blocks=True)
    torch.cuda.synchronize()
    r = raw.cpu().numpy().view(dxt1.CLUSTER_DTYPE).reshape(-1)
    sel = sel.cpu().numpy()
    flags = (oracle.DXT1_PERCEPTUAL if perceptual else 0) | oracle.DXT1_ALPHA_BLOCKS
    alpha_blocks = 0
    for c, p in enumerate(parts):
        osel, ores = oracle.dxt1_cluster(p, 4, flags)
        lo, hi = int(r["lo_hi"][c] & 0xFFFF), int(r["lo_hi"][c] >> 16)
        s = sel[ofs[c]:ofs[c + 1]]
        assert int(r["error"][c]) == ores.error, (c, len(p))
        assert (lo, hi) == (ores.low, ores.high), c
        assert np.array_equal(s, osel), c
        assert ((int(r["flags"][c]) >> 1) & 1) == ores.alpha_block, c
        alpha_blocks += ores.alpha_block
    print("3-colour clusters", alpha_blocks, "of", len(parts), flush=True)


def test_clusters_with_transparent_texels_match_oracle(gpu):
    # DXT1A (qdxt1's clusters with a texel below the threshold): colours from
    # the opaque texels only, 3-colour blocks, transparent texels on selector 3
    rng = np.random.default_rng(33)
    parts = clusters(50, [16, 48, 200, 700, 1500, 3000, 5000])
    for k, p in enumerate(parts):
        p = p.copy()
        p[:, 3] = 255
        p[rng.random(len(p)) < 0.3, 3] = rng.integers(0, 128)
        parts[k] = p
    allt = parts[0].copy()
    allt[:, 3] = 0                                                              # no opaque texel
    one = np.repeat(parts[1][:1], 64, axis=0)
    one[::3, 3] = 5                                                             # one opaque colour
    noisy = rng.integers(0, 256, (6000, 4), dtype=np.uint8)                     # global-memory pass
    parts += [allt, one, noisy]
    px = np.concatenate(parts)
    ofs = np.concatenate([[0], np.cumsum([len(p) for p in parts])]).astype(np.int32)
    t = torch.from_numpy(px).cuda()
    o = torch.from_numpy(ofs).cuda()
    out, sel = dxt1.encode_clusters_device(t, o, True, True, alpha_blocks=True, alpha_threshold=128)
    torch.cuda.synchronize()
    r = out.cpu().numpy().view(dxt1.CLUSTER_DTYPE).reshape(-1)
    sel = sel.cpu().numpy()
    for c, p in enumerate(parts):
        have = bool((p[:, 3] < 128).any())
        flags = oracle.DXT1_PERCEPTUAL | oracle.DXT1_ALPHA_BLOCKS | (oracle.DXT1_HAVE_ALPHA if have else 0) | \
            oracle.dxt1_threshold(128)
        osel, ores = oracle.dxt1_cluster(p, 4, flags)
        lo, hi = int(r["lo_hi"][c] & 0xFFFF), int(r["lo_hi"][c] >> 16)
        assert int(r["error"][c]) == ores.error, (c, len(p))
        assert (lo, hi) == (ores.low, ores.high), c
        assert np.array_equal(sel[ofs[c]:ofs[c + 1]], osel), c
        assert ((int(r["flags"][c]) >> 1) & 1) == ores.alpha_block, c


@pytest.mark.parametrize("uber", [False, True])
@pytest.mark.parametrize("around", [512, 1024, 2048, 4096])
def test_cluster_class_edges_match_oracle(gpu, around, uber):
    """Texel counts on either side of each size class's limit, as runs of few
    colours, as all-different colours and as one colour with an odd one out:
    the sorted and the hashed colour sets, one to eight waves per cluster, and
    colour counts off the 32-wide tiles of the scoring."""
    rng = np.random.default_rng(around + uber)
    parts = []
    for n in (around - 1, around, around + 1, around + 33):
        runs = np.repeat(rng.integers(0, 256, (n // 37 + 1, 4), dtype=np.uint8), 37, axis=0)[:n]
        parts += [runs, rng.integers(96, 160, (n, 4), dtype=np.uint8)]
        flat = np.repeat(runs[:1], n, axis=0)
        flat[n // 2, 1] ^= 0x40
        parts.append(flat)
    if around == 4096:
        few = rng.integers(0, 16, (30000, 4), dtype=np.uint8) * 16                  # every colour of a 16^3 cube
        parts += [few, np.concatenate([few, np.full((1, 4), 7, np.uint8)])]         # 4,096 and 4,097 colours
    px = np.concatenate(parts)
    ofs = np.concatenate([[0], np.cumsum([len(p) for p in parts])]).astype(np.int32)
    print("clusters around", around, "uber", uber, flush=True)
    raw, sel = dxt1.encode_clusters_device(torch.from_numpy(px).cuda(), torch.from_numpy(ofs).cuda(), True,
                                           alpha_blocks=uber)
    torch.cuda.synchronize()
    r = raw.cpu().numpy().view(dxt1.CLUSTER_DTYPE).reshape(-1)
    sel = sel.cpu().numpy()
    flags = oracle.DXT1_PERCEPTUAL | (oracle.DXT1_ALPHA_BLOCKS if uber else 0)
    for c, p in enumerate(parts):
        osel, ores = oracle.dxt1_cluster(p, 4, flags)
        assert r["nunique"][c] == len(np.unique(p[:, :3], axis=0)), c
        assert int(r["error"][c]) == ores.error, (c, len(p))
        assert (int(r["lo_hi"][c] & 0xFFFF), int(r["lo_hi"][c] >> 16)) == (ores.low, ores.high), c
        assert np.array_equal(sel[ofs[c]:ofs[c + 1]], osel), c
