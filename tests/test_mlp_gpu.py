"""Learned DXT1 endpoint proposal on the GPU against the oracle
(oracle/mlp.py): features, the strided GEMM, forward/backward gradients of the
training kernels, the bfloat16 matrix-core inference, the exact refinement
error, and an ablation showing what the trained network gains."""
import ctypes as C

import numpy as np
import pytest
import torch

from oracle import mlp as omlp
from crunch2_amd import dxt1, learned, texture
from crunch2_amd._lib import check, lib
from tests.hc_cases import blocks_from_texture

pytestmark = pytest.mark.gpu

W = np.array([8, 25, 1], np.int64)


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def test_features(gpu):
    blocks = blocks_from_texture(64, 1)
    f = learned.features(dev(blocks)).cpu().numpy()
    assert np.allclose(f, omlp.features(blocks), atol=2e-6)


@pytest.mark.parametrize("M,N,K,ks,ra,rb", [(1, 1, 1, 1, 0, 0), (70, 130, 57, 1, 1, 1), (128, 7, 5000, 8, 0, 0),
                                           (33, 128, 128, 1, 0, 1), (1, 128, 3000, 4, 0, 0)])
def test_gemm(gpu, M, N, K, ks, ra, rb):
    print("gemm", M, N, K, ks, flush=True)
    rng = np.random.default_rng(M * 7 + N)
    A = rng.standard_normal((K, M)).astype(np.float32)     # stored transposed: A(m, k) = A[k, m]
    B = rng.standard_normal((K, N)).astype(np.float32)
    C = torch.zeros((M, N), dtype=torch.float32, device="cuda")
    learned.gemm(M, N, K, dev(A), 1, M, dev(B), N, 1, C, N, round_a=ra, round_b=rb, ksplit=ks)
    a = omlp.bf16(A) if ra else A
    b = omlp.bf16(B) if rb else B
    ref = a.T.astype(np.float64) @ b.astype(np.float64)
    assert np.allclose(C.cpu().numpy(), ref, rtol=1e-4, atol=1e-3 * np.sqrt(K))


def training_batch(n, seed):
    blocks = dxt1.image_blocks(texture.synth(128, 128, seed, texture.RGB))[:n]
    rng = np.random.default_rng(seed)
    t = rng.random((len(blocks), 6)).astype(np.float32)
    return blocks, t


def test_gradients_match_oracle(gpu):
    blocks, t = training_batch(512, 3)
    theta = omlp.init_params(7)
    tr = learned.Trainer(dev(theta))
    x = learned.features(dev(blocks))
    loss, g = tr.gradients(x, dev(t))
    torch.cuda.synchronize()
    ref_loss, ref_g = omlp.loss_and_grads(theta, x.cpu().numpy(), t)
    g = g.cpu().numpy()
    print("loss", float(loss.item()), ref_loss, flush=True)
    assert abs(float(loss.item()) - ref_loss) <= 1e-4 * max(1.0, abs(ref_loss))
    cos = float(g @ ref_g / (np.linalg.norm(g) * np.linalg.norm(ref_g)))
    rel = np.abs(g - ref_g).max() / np.abs(ref_g).max()
    print("gradient cosine %.8f max rel %.2e" % (cos, rel), flush=True)
    assert cos > 0.99999 and rel < 1e-3


def test_gradients_with_given_labels_match_oracle(gpu):
    blocks, t = training_batch(512, 8)
    theta = omlp.init_params(9)
    lab = (np.random.default_rng(8).random(len(blocks)) < 0.3).astype(np.float32)
    tr = learned.Trainer(dev(theta))
    x = learned.features(dev(blocks))
    loss, g = tr.gradients(x, dev(t), dev(lab))
    torch.cuda.synchronize()
    ref_loss, ref_g = omlp.loss_and_grads(theta, x.cpu().numpy(), t, labels=lab)
    g = g.cpu().numpy()
    assert abs(float(loss.item()) - ref_loss) <= 1e-4 * max(1.0, abs(ref_loss))
    cos = float(g @ ref_g / (np.linalg.norm(g) * np.linalg.norm(ref_g)))
    assert cos > 0.99999 and np.abs(g - ref_g).max() / np.abs(ref_g).max() < 1e-3
    # the labels reach the confidence output: its bias gradient changes with them
    _, g2 = tr.gradients(x, dev(t), dev(1.0 - lab))
    assert abs(float(g2[-1].item()) - float(g[-1])) > 1e-6


@pytest.mark.parametrize("n", [1, 31, 33, 63, 65, 8192, 8193, 16385])
def test_gradients_at_tile_edges(gpu, n):
    """Row counts around the 32- and 64-row steps, the switch between them and
    the largest grid, against the oracle; the same batch twice gives the same
    bits.  The error is that of activations that round to the other bfloat16
    neighbour (2^-9 of one of 128 terms), so the bounds are those of the other
    gradient tests."""
    print("gradients", n, flush=True)
    blocks = dxt1.image_blocks(texture.synth(520, 520, n, texture.RGB))[:n]
    t = np.random.default_rng(n).random((n, 6)).astype(np.float32)
    theta = omlp.init_params(n)
    tr = learned.Trainer(dev(theta))
    x = learned.features(dev(blocks))
    loss, g = tr.gradients(x, dev(t))
    one = (float(loss.item()), g.cpu().numpy().copy())
    ref_loss, ref_g = omlp.loss_and_grads(theta, x.cpu().numpy(), t)
    assert abs(one[0] - ref_loss) <= 1e-4 * max(1.0, abs(ref_loss))
    cos = float(one[1] @ ref_g / (np.linalg.norm(one[1]) * np.linalg.norm(ref_g)))
    assert cos > 0.99999 and np.abs(one[1] - ref_g).max() / np.abs(ref_g).max() < 1e-3
    loss, g = tr.gradients(x, dev(t))
    assert float(loss.item()) == one[0] and np.array_equal(g.cpu().numpy(), one[1])


def test_inference_matches_oracle(gpu):
    blocks, _ = training_batch(700, 4)
    theta = omlp.init_params(11)
    y = learned.infer(dev(theta), dev(blocks)).cpu().numpy()
    ref, _ = omlp.forward(theta, omlp.features(blocks))
    d = np.abs(y[:, :7] - ref)
    print("inference max abs diff %.3e" % d.max(), flush=True)
    assert d.max() < 2e-2 and np.median(d) < 1e-3


def np_block_error(px, c0, c1):
    def ex(c):
        r, g, b = (c >> 11) & 31, (c >> 5) & 63, c & 31
        return np.array([(r << 3) | (r >> 2), (g << 2) | (g >> 4), (b << 3) | (b >> 2)], np.int64)
    p0, p1 = ex(int(c0)), ex(int(c1))
    if c0 > c1:
        pal = [p0, p1, (2 * p0 + p1) // 3, (p0 + 2 * p1) // 3]
    else:
        pal = [p0, p1, (p0 + p1) // 2, np.zeros(3, np.int64)]
    d = np.stack([(((px[:, :3].astype(np.int64) - q) ** 2) * W).sum(1) for q in pal], 1)
    return int(d.min(1).sum())


def test_refinement_is_exact_and_locally_optimal(gpu):
    blocks, _ = training_batch(300, 5)
    rng = np.random.default_rng(6)
    y = np.zeros((len(blocks), 8), np.float32)
    y[:, :6] = rng.random((len(blocks), 6))
    out = learned.refine(dev(blocks), dev(y), max_iters=64).cpu().numpy().view(np.uint32)
    for b in range(len(blocks)):
        c0, c1 = out[b, 0] & 0xFFFF, out[b, 0] >> 16
        assert out[b, 2] == np_block_error(blocks[b], c0, c1)
        if out[b, 3] < 64:       # converged: no single +-1 channel step improves
            for ci, c in enumerate((c0, c1)):
                for sh, bits in ((11, 5), (5, 6), (0, 5)):
                    v = (int(c) >> sh) & ((1 << bits) - 1)
                    for d in (-1, 1):
                        if 0 <= v + d < (1 << bits):
                            nc = (int(c) & ~(((1 << bits) - 1) << sh)) | ((v + d) << sh)
                            e0, e1 = (nc, c1) if ci == 0 else (c0, nc)
                            e0, e1 = max(e0, e1), min(e0, e1)
                            assert np_block_error(blocks[b], e0, e1) >= out[b, 2]


def train_small(seed=0, steps=300, n=262144, batch=8192):
    imgs = [texture.synth(512, 512, 100 + s, texture.RGB) for s in range(n // 16384)]
    blocks = np.concatenate([dxt1.image_blocks(im) for im in imgs])
    tb = dev(blocks)
    t, _ = learned.plain_targets(tb)
    x = learned.features(tb)
    tr = learned.Trainer(seed=seed, lr=2e-3)
    g = torch.Generator(device="cuda").manual_seed(seed)
    for s in range(steps):
        idx = torch.randint(0, x.shape[0], (batch,), device="cuda", generator=g)
        tr.step(x[idx].contiguous(), t[idx].contiguous())
    return tr


def layered_gradients(theta, X, T, labels):
    """The loss and gradient layer by layer through the layers' own entry points."""
    n, o, N, H, K = X.shape[0], learned.OFFSETS, learned.N_IN, learned.N_H, learned.N_OUT
    new = lambda *s: torch.zeros(s, dtype=torch.float32, device="cuda")
    p = lambda t, ofs=0: C.c_void_p(t.data_ptr() + 4 * ofs if t is not None else 0)
    s, L, mm = C.c_void_p(torch.cuda.current_stream().cuda_stream), lib(), learned.gemm
    Z1, A1, Z2, A2, dA, dZ, Y, dY = new(n, H), new(n, H), new(n, H), new(n, H), new(n, H), new(n, H), new(n, K), new(n, K)
    g, loss, ones = torch.zeros_like(theta), new(1), torch.ones(1, device="cuda")
    mm(n, H, N, X, N, 1, theta, H, 1, Z1, H, round_a=True, round_b=True, b_ofs=o["W1"])
    check(L.crn2_mlp_bias_act_device(p(Z1), p(A1), p(theta, o["b1"]), n, H, 1, s))
    mm(n, H, H, A1, H, 1, theta, H, 1, Z2, H, round_b=True, b_ofs=o["W2"])
    check(L.crn2_mlp_bias_act_device(p(Z2), p(A2), p(theta, o["b2"]), n, H, 1, s))
    mm(n, K, H, A2, H, 1, theta, K, 1, Y, K, round_b=True, b_ofs=o["W3"])
    check(L.crn2_mlp_bias_act_device(p(Y), p(Y), p(theta, o["b3"]), n, K, 0, s))
    check(L.crn2_mlp_loss_device(p(Y), p(T), p(labels), n, p(dY), p(loss), s))
    ks = max(1, min(64, n // 1024))
    mm(H, K, n, A2, 1, H, dY, K, 1, g, K, ksplit=ks, c_ofs=o["W3"])
    mm(1, K, n, ones, 0, 0, dY, K, 1, g, K, ksplit=ks, c_ofs=o["b3"])
    mm(n, H, K, dY, K, 1, theta, 1, K, dA, H, round_b=True, b_ofs=o["W3"])
    check(L.crn2_mlp_gelu_back_device(p(dA), p(Z2), p(dZ), n * H, s))
    mm(H, H, n, A1, 1, H, dZ, H, 1, g, H, ksplit=ks, c_ofs=o["W2"])
    mm(1, H, n, ones, 0, 0, dZ, H, 1, g, H, ksplit=ks, c_ofs=o["b2"])
    mm(n, H, H, dZ, H, 1, theta, 1, H, dA, H, round_b=True, b_ofs=o["W2"])
    check(L.crn2_mlp_gelu_back_device(p(dA), p(Z1), p(dZ), n * H, s))
    mm(N, H, n, X, 1, N, dZ, H, 1, g, H, round_a=True, ksplit=ks, c_ofs=o["W1"])
    mm(1, H, n, ones, 0, 0, dZ, H, 1, g, H, ksplit=ks, c_ofs=o["b1"])
    return loss, g


@pytest.mark.parametrize("n", [1, 300, 5000])
@pytest.mark.parametrize("labelled", [False, True])
def test_layers_match_the_fused_gradient(gpu, n, labelled):
    """The layers' entry points and the fused kernel compute the same loss and
    gradient.  Both sum in float32 in other orders; an activation near a
    bfloat16 step can round to either neighbour, which moves one of its 128
    terms by 2^-9 of itself: 2^-9 / 128 of the whole, for a few rows, or 1.5e-5
    for one row alone."""
    print("layers", n, labelled, flush=True)
    blocks = dxt1.image_blocks(texture.synth(300, 300, n, texture.RGB))[:n]
    rng = np.random.default_rng(n)
    t, lab = dev(rng.random((n, 6)).astype(np.float32)), dev(rng.integers(0, 2, n).astype(np.float32))
    theta = dev(omlp.init_params(n))
    x = learned.features(dev(blocks))
    loss, g = learned.Trainer(theta).gradients(x, t, lab if labelled else None)
    rloss, rg = layered_gradients(theta, x, t, lab if labelled else None)
    assert abs(float(loss.item()) - float(rloss.item())) <= 2e-5 * max(1.0, abs(float(rloss.item())))
    assert float((g - rg).norm() / rg.norm()) <= 2e-5


def _pair_errors(px, e):
    """Errors of many endpoint pairs e (k x 2 x 3, 5:6:5 components) on one
    block's texels (16 x 3), the pair in either order."""
    w = np.array([1 << 11, 1 << 5, 1])
    c = (e * w).sum(-1)
    hi = np.where((c[:, 0] >= c[:, 1])[:, None], e[:, 0], e[:, 1])
    lo = np.where((c[:, 0] >= c[:, 1])[:, None], e[:, 1], e[:, 0])

    def ex(v):
        return np.stack([v[:, 0] << 3 | v[:, 0] >> 2, v[:, 1] << 2 | v[:, 1] >> 4, v[:, 2] << 3 | v[:, 2] >> 2], 1)
    p, q = ex(hi), ex(lo)
    four = (c[:, 0] != c[:, 1])[:, None]
    pal = np.stack([p, q, np.where(four, (2 * p + q) // 3, (p + q) // 2), np.where(four, (p + 2 * q) // 3, 0)], 1)
    d = ((px[None, None] - pal[:, :, None]) ** 2 * W).sum(-1)
    return d.min(1).sum(1)


def _best_move(px, e, moves, err):
    f = e[None] + moves
    ok = ((f >= 0) & (f <= np.array([31, 63, 31]))).all((1, 2))
    er = np.where(ok, _pair_errors(px, np.clip(f, 0, 63)), 1 << 40)
    k = int(er.argmin())
    return (k, int(er[k])) if er[k] < err else (None, err)


@pytest.mark.parametrize("kind", ["texture", "near flat", "dark", "noise"])
def test_polish_takes_the_first_best_lattice_move(gpu, kind):
    """The polish against its own definition in numpy: from the unpolished
    result (in both orders of the endpoints), up to four times the first of the
    smallest errors among the 728 moves, then single steps while they help;
    near-flat blocks have candidates with equal endpoints."""
    print("polish", kind, flush=True)
    rng = np.random.default_rng(len(kind))
    n = 130
    if kind == "texture":
        blocks = dxt1.image_blocks(texture.synth(64, 64, 5, texture.RGB))[:n].copy()
    else:
        spread, top = {"near flat": (6, 250), "dark": (12, 13), "noise": (256, 1)}[kind]
        blocks = (rng.integers(0, top, (n, 1, 4)) + rng.integers(0, spread, (n, 16, 4))).clip(0, 255).astype(np.uint8)
    t = dev(blocks)
    start = learned.refine(t, None, 16, learned.START_BOX).cpu().numpy().view(np.uint32)
    got = learned.refine(t, None, 16, learned.START_BOX | learned.POLISH).cpu().numpy().view(np.uint32)
    ms = np.arange(729)
    box = np.stack([(ms // 3 ** k) % 3 - 1 for k in range(6)], 1).reshape(-1, 2, 3)[np.arange(729) != 364]
    one = np.array([[s, k, d] for s in range(2) for k in range(3) for d in (-1, 1)])
    steps = np.zeros((12, 2, 3), int)
    steps[np.arange(12), one[:, 0], one[:, 1]] = one[:, 2]
    moved = 0
    for i in range(n):
        px = blocks[i, :, :3].astype(np.int64)
        best = int(start[i, 2])
        results = []
        for order in (0, 1):          # the start's endpoints in either order: only ties tell them apart
            c = [int(start[i, 0] & 0xFFFF), int(start[i, 0] >> 16)]
            e = np.array([[v >> 11, v >> 5 & 63, v & 31] for v in (c[::-1] if order else c)])
            err = best
            for _ in range(4):
                if not err:
                    break
                k, err = _best_move(px, e, box, err)
                if k is None:
                    break
                e = e + box[k]
                for _ in range(16):
                    k, err = _best_move(px, e, steps, err)
                    if k is None:
                        break
                    e = e + steps[k]
            words = (e * np.array([1 << 11, 1 << 5, 1])).sum(-1)
            results.append((int(words.max()) | int(words.min()) << 16, err))
        assert (int(got[i, 0]), int(got[i, 2])) in results, (i, results)
        moved += int(got[i, 2]) < best
    assert kind == "dark" or moved > 5


@pytest.mark.parametrize("starts", [learned.START_NET, learned.ENCODE_STARTS])
def test_refinement_paths_agree_at_the_switch(gpu, starts):
    """The largest call of one wavefront per block (57,344 blocks) and the
    smallest of one lane per block give the same for the same blocks."""
    print("refinement switch", starts, flush=True)
    t = dev(dxt1.image_blocks(texture.synth(1032, 1024, 13, texture.RGB))[:57345])
    y = learned.infer(dev(np.load("crunch2_amd/data/dxt1_proposal.npy")), t)
    lanes = learned.refine(t, y, learned.ENCODE_ITERS, starts)
    waves = learned.refine(t[:57344], y[:57344], learned.ENCODE_ITERS, starts)
    assert torch.equal(lanes[:57344], waves)


@pytest.mark.parametrize("starts", [learned.START_NET, learned.ENCODE_STARTS])
def test_refinement_paths_agree(gpu, starts):
    """A call of 65,537 blocks (one lane per block, the polish on its own) gives
    what calls of fewer (one wavefront per block) give for the same blocks."""
    print("refinement paths", starts, flush=True)
    t = dev(dxt1.image_blocks(texture.synth(1032, 1024, 12, texture.RGB))[:65537])
    y = learned.infer(dev(np.load("crunch2_amd/data/dxt1_proposal.npy")), t)
    whole = learned.refine(t, y, learned.ENCODE_ITERS, starts)
    parts = [learned.refine(t[a:b], y[a:b], learned.ENCODE_ITERS, starts) for a, b in ((0, 65536), (65536, 65537))]
    assert torch.equal(whole, torch.cat(parts))


def test_training_gains_over_untrained_and_box_start(gpu):
    """Ablation on held-out blocks.  The method without the network refines
    from the block's brightest/darkest texels; with it, the refinement also
    starts from the network's proposal and keeps the better.  The trained
    network must lower the total error and raise the share of blocks that
    reach the plain search's error; an untrained network must gain less."""
    tr = train_small(steps=1500)
    test = dev(dxt1.image_blocks(texture.synth(256, 256, 999, texture.RGB)))
    plain = dxt1.encode_blocks_device(test, dxt1.UBER, learned.LABEL_FLAGS)
    perr, _ = learned.block_errors(test, plain.view(torch.int32).reshape(-1, 6)[:, 2].contiguous())
    runs = {
        "box only": learned.refine(test, None, 8, learned.START_BOX),
        "untrained + box": learned.refine(test, learned.infer(learned.init_params(0), test), 8,
                                          learned.START_NET | learned.START_BOX),
        "trained + box": learned.refine(test, learned.infer(tr.theta, test), 8,
                                        learned.START_NET | learned.START_BOX),
        "trained only": learned.refine(test, learned.infer(tr.theta, test), 8, learned.START_NET),
    }
    res = {}
    for k, r in runs.items():
        res[k] = (float(r[:, 2].double().sum()), float((r[:, 2] <= perr).float().mean()))
        print(k, "total error %.5g, blocks at or below plain %.4f" % res[k], flush=True)
    assert res["trained + box"][0] < res["box only"][0]
    assert res["trained + box"][1] > res["box only"][1]
    gain_trained = res["box only"][0] - res["trained + box"][0]
    gain_untrained = res["box only"][0] - res["untrained + box"][0]
    assert gain_trained > gain_untrained


def test_guarded_encode_never_worse_than_plain(gpu):
    tr = train_small(steps=100)
    test = dev(dxt1.image_blocks(texture.synth(128, 128, 555, texture.RGB)))
    ends, sels, errs, nplain = learned.encode(tr.theta, test, guarded=True)
    plain = dxt1.encode_blocks_device(test, dxt1.UBER, learned.LABEL_FLAGS)
    perr, _ = learned.block_errors(test, plain.view(torch.int32).reshape(-1, 6)[:, 2].contiguous())
    assert nplain == len(test)
    assert bool((errs <= perr).all())
    e2, s2 = learned.block_errors(test, ends)
    assert bool((e2 == errs).all()) and bool((s2 == sels).all())
