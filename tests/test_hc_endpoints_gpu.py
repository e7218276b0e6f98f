"""dxt_hc colour endpoint codebook on the GPU (crn2_hc_color_endpoints_device)
against the oracle: cluster endpoints after the refiner, cluster colours and
every block's selector word, bit for bit."""
import numpy as np
import pytest
import torch

import oracle
from crunch2_amd import hc
from tests.hc_endpoint_cases import clusters

pytestmark = pytest.mark.gpu


def run_gpu(px, ofs, bc, blocks, w, enc, perceptual):
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    ends, cv, bsel, ne = hc.color_endpoints(d(px), d(ofs.astype(np.int32)), d(bc.view(np.int32)), d(blocks), d(w),
                                            d(enc), perceptual)
    torch.cuda.synchronize()
    return ends.cpu().numpy().view(np.uint32), cv.cpu().numpy(), bsel.cpu().numpy().view(np.uint64), ne


@pytest.mark.parametrize("seed,perceptual,side,k", [(0, True, 128, 48), (1, False, 128, 48), (2, True, 256, 96)])
def test_endpoint_codebook_matches_oracle(gpu, seed, perceptual, side, k):
    """Every cluster, including those of more than 4,096 distinct colours
    (searched with their colour set in global memory), bit for bit."""
    print("hc endpoints seed", seed, "perceptual", perceptual, "side", side, "clusters", k, flush=True)
    px, ofs, bc, blocks, w, enc = clusters(side=side, k=k, seed=seed)
    ends, cv, bsel, ne = run_gpu(px, ofs, bc, blocks, w, enc, perceptual)
    rends, rcv, rbsel = oracle.hc_color_endpoints(px, ofs, bc, blocks, w, enc, perceptual)
    big = np.array([len(np.unique(px[ofs[c]:ofs[c + 1]].view(np.uint32))) > 4096 for c in range(k)])
    print("clusters beyond 4096 colours:", int(big.sum()), flush=True)
    assert ne == 0
    assert np.array_equal(cv, rcv)
    assert np.array_equal(ends, rends), np.nonzero(ends != rends)[0][:10]
    inb = bc != 0xFFFFFFFF
    assert np.array_equal(bsel[inb], rbsel[inb])
    assert (bsel[~inb] == 0).all()


@pytest.mark.parametrize("seed,side,k", [(0, 128, 40), (1, 256, 64)])
def test_alpha_endpoint_codebook_matches_oracle(gpu, seed, side, k):
    from tests.hc_endpoint_cases import alpha_clusters
    print("hc alpha endpoints seed", seed, "side", side, "clusters", k, flush=True)
    vals, ofs, bc, blocks, enc = alpha_clusters(side=side, k=k, seed=seed)
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    ends, av, rv, bsel = hc.alpha_endpoints(d(vals), d(ofs.astype(np.int32)), d(bc.view(np.int32)), d(blocks), d(enc))
    torch.cuda.synchronize()
    ends, av, rv = ends.cpu().numpy().view(np.uint32), av.cpu().numpy(), rv.cpu().numpy()
    bsel = bsel.cpu().numpy().view(np.uint64)
    rends, rav, rrv, rbsel = oracle.hc_alpha_endpoints(vals, ofs, bc, blocks, enc)
    assert np.array_equal(av, rav)
    assert np.array_equal(ends, rends), np.nonzero(ends != rends)[0][:10]
    assert np.array_equal(rv, rrv)
    assert np.array_equal(bsel, rbsel)


def _one_cluster_each(sizes):
    ofs = np.zeros(len(sizes) + 1, np.uint32)
    ofs[1:] = np.cumsum(sizes)
    blocks = np.zeros((2, 16, 4), np.uint8)
    return ofs, np.full(2, 0xFFFFFFFF, np.uint32), blocks


@pytest.mark.parametrize("sizes", [(1, 2, 3, 5, 63, 65, 257, 1023, 4097), (300001,)])
@pytest.mark.parametrize("what", ["flat", "two", "noise"])
def test_refiner_sums_any_size(gpu, sizes, what):
    """The refiners' parallel sums give the start of the sums in texel order:
    clusters of any texel count, flat ones (the singular system of one colour
    on a middle selector, whose sums round once per texel) and noisy ones."""
    print("hc refiner", what, sizes, flush=True)
    rng = np.random.default_rng(len(sizes))
    ofs, bc, blocks = _one_cluster_each(sizes)
    px = np.full((ofs[-1], 4), 255, np.uint8)
    for a, b in zip(ofs[:-1], ofs[1:]):
        if what == "noise":
            px[a:b, :3] = np.clip(rng.integers(0, 256, 3) + rng.normal(0, 9, (b - a, 3)), 0, 255)
            px[a:b, :3] &= 0xFC if b - a > 5000 else 0xFF     # few enough distinct colours for the oracle
        else:
            px[a:b, :3] = rng.integers(0, 256, 3)
            if what == "two":
                px[a + (b - a) // 3:b, :3] = rng.integers(0, 256, 3)
    w, enc = np.ones(2, np.float32), np.zeros(2, np.uint8)
    ends, cv, _, ne = run_gpu(px, ofs, bc, blocks, w, enc, True)
    rends, rcv, _ = oracle.hc_color_endpoints(px, ofs, bc, blocks, w, enc, True)
    assert ne == 0
    assert np.array_equal(cv, rcv)
    assert np.array_equal(ends, rends), np.nonzero(ends != rends)[0][:10]
    vals, av = np.ascontiguousarray(px[:, 1]), blocks[:, :, 3].copy()
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    got = hc.alpha_endpoints(d(vals), d(ofs.astype(np.int32)), d(bc.view(np.int32)), d(av), d(enc))
    torch.cuda.synchronize()
    ref = oracle.hc_alpha_endpoints(vals, ofs, bc, av, enc)
    assert np.array_equal(got[0].cpu().numpy().view(np.uint32), ref[0])
    assert np.array_equal(got[1].cpu().numpy(), ref[1]) and np.array_equal(got[2].cpu().numpy(), ref[2])


# Two neighbouring values, how often each, and the step j: the mean of their
# float32 values over 255 is exactly j / 256 (of the last, 43 / 64 too).
ON_THE_LINE = [(164, 466, 257, 165), (138, 916, 771, 139), (216, 1430, 257, 217), (171, 2105, 1028, 172)]


@pytest.mark.parametrize("k", [1, 3])
@pytest.mark.parametrize("far", [0, 255])
def test_refiner_start_on_a_line_of_the_cut(gpu, k, far):
    """The best block gives both values one end and the far one the other, so
    that end's least-squares start lies on a line of its cut: the bound of the
    parallel sums reaches over it, and the sums are taken in texel order.  The
    endpoints are the oracle's."""
    print("refiner start on the line", k, far, flush=True)
    rng = np.random.default_rng(k + far)
    parts = []
    for v, a, b, j in ON_THE_LINE:
        x = [float(np.float32(u) / np.float32(255.0)) for u in (v, v + 1)]
        assert (a * x[0] + b * x[1]) * 256 == (a + b) * j      # (exact in doubles)
        for _ in range(3):
            parts.append(rng.permutation(np.array([v] * (a * k) + [v + 1] * (b * k) + [far] * 70, np.uint8)))
    ofs, bc, blocks = _one_cluster_each([len(v) for v in parts])
    vals = np.concatenate(parts)
    av, enc = blocks[:, :, 3].copy(), np.zeros(2, np.uint8)
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    got = hc.alpha_endpoints(d(vals), d(ofs.astype(np.int32)), d(bc.view(np.int32)), d(av), d(enc))
    torch.cuda.synchronize()
    ref = oracle.hc_alpha_endpoints(vals, ofs, bc, av, enc)
    for c, v in enumerate(parts):     # one end for the two values, the other for the far one
        near = ref[1][c].astype(int)
        assert sorted(near[[0, 7]])[0 if far else 1] in (v[v != far].min(), v[v != far].max()) and far in near[[0, 7]]
    assert np.array_equal(got[0].cpu().numpy().view(np.uint32), ref[0])
    assert np.array_equal(got[1].cpu().numpy(), ref[1]) and np.array_equal(got[2].cpu().numpy(), ref[2])
    # the same as grey colours (cut to 32 and 64 steps)
    px = np.full((len(vals), 4), 255, np.uint8)
    px[:, :3] = vals[:, None]
    w = np.ones(2, np.float32)
    ends, cv, _, ne = run_gpu(px, ofs, bc, blocks, w, enc, True)
    rends, rcv, _ = oracle.hc_color_endpoints(px, ofs, bc, blocks, w, enc, True)
    assert ne == 0 and np.array_equal(cv, rcv) and np.array_equal(ends, rends)
