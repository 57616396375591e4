"""AMP discriminator update on the GPU against the float64 oracle (ksim/task/amp.py:360-545)."""
import numpy as np
import pytest
import torch

from oracle import amp as oamp
from oracle import ppo_update as oup

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
GRAD_TOL = 2e-4   # fp32 products against float64, relative to the largest entry of each gradient
LOSS_TOL = 1e-5


def _params(dims, seed):
    rng = np.random.default_rng(seed)
    ws = [(rng.normal(size=(o, i)) / np.sqrt(i)).astype(np.float32) for i, o in zip(dims[:-1], dims[1:])]
    bs = [(rng.normal(size=o) * 0.1).astype(np.float32) for o in dims[1:]]
    return ws, bs


def _check(disc, ws, bs, real, sim, coef, act):
    losses = disc.disc_loss_grad(torch.tensor(real, device=DEV), torch.tensor(sim, device=DEV), coef).cpu().numpy()
    want_l, want_g = oamp.disc_loss_and_grads(ws, bs, real, sim, coef, act=act)
    np.testing.assert_allclose(losses, want_l, rtol=LOSS_TOL, atol=1e-6)
    for l, ((gw, gb), (ww, wb)) in enumerate(zip(disc.parameters(gradients=True), want_g)):
        for name, got, want in (("weight", gw, ww), ("bias", gb, wb)):
            err = np.abs(got.cpu().numpy() - want).max() / max(np.abs(want).max(), 1e-6)
            assert err <= GRAD_TOL, f"layer {l} {name}: {err:.2e}"
    return losses


@pytest.mark.parametrize("act,dims,dtype", [("elu", [37, 96, 64, 1], "f32"), ("tanh", [12, 50, 1], "f32"), ("relu", [20, 33, 17, 1], "f32"),
                                            ("elu", [5, 1], "f32"), ("elu", [24, 128, 128, 1], "bf16")])
def test_discriminator_loss_gradient_matches_oracle(act, dims, dtype):
    """Squared-error terms and the gradient penalty (which differentiates the network twice); ragged widths, a linear
    network, and a bf16 network (the update itself runs on the fp32 master weights)."""
    from ksim_amd.mlp import MLP

    ws, bs = _params(dims, seed=len(dims) * 7 + dims[0])
    disc = MLP(ws, bs, activation=act, dtype=dtype)
    disc.train_init()
    rng = np.random.default_rng(5)
    real = rng.normal(size=(6, 11, dims[0])).astype(np.float32)
    sim = rng.normal(size=(4, 9, dims[0])).astype(np.float32)
    l1 = _check(disc, ws, bs, real, sim, 10.0, act)
    assert l1[2] > 1e-3
    # a second call on fewer rows reuses the workspace and overwrites the gradients; no penalty this time
    l0 = _check(disc, ws, bs, real[:2], sim[:1], 0.0, act)
    assert l0[2] == 0.0


@pytest.mark.parametrize("dims", [[30, 64, 1], [30, 256, 130, 1]])
def test_discriminator_many_rows_split_reduction(dims):
    """Enough frames that the weight-gradient products cut their row range into slices; with layers of 128 units and more
    they run on the wide tiles, the bias gradients summed in the same pass (a width that ends inside a tile included)."""
    from ksim_amd.mlp import MLP

    ws, bs = _params(dims, seed=3)
    disc = MLP(ws, bs, activation="elu", dtype="f32")
    disc.train_init()
    rng = np.random.default_rng(8)
    real = rng.normal(size=(32, 100, 30)).astype(np.float32)
    sim = rng.normal(size=(32, 100, 30)).astype(np.float32)
    _check(disc, ws, bs, real, sim, 10.0, "elu")


@pytest.mark.parametrize("act,dims,real_rows,sim_rows", [("elu", [17, 320, 272, 31, 1], 16, 1), ("tanh", [16, 300, 1], 15, 17), ("elu", [48, 16, 1], 33, 0),
                                                         ("tanh", [9, 130, 64, 50, 1], 1, 47), ("relu", [33, 321, 40, 1], 17, 16), ("elu", [321, 64, 1], 5, 33)])
def test_discriminator_rows_at_the_edges_of_their_launch(act, dims, real_rows, sim_rows):
    """Sixteen rows and sixteen columns at a time, up to 320 wide, in the launch that takes a frame through the whole chain: ragged ends of both,
    reductions that end inside a step, more columns than one pass of the wavefronts, three hidden layers, and the first width of the general route."""
    from ksim_amd.mlp import MLP

    ws, bs = _params(dims, seed=sum(dims))
    disc = MLP(ws, bs, activation=act, dtype="f32")
    disc.train_init()
    rng = np.random.default_rng(real_rows)
    real, sim = (rng.normal(size=(n, 1, dims[0])).astype(np.float32) for n in (real_rows, sim_rows))
    _check(disc, ws, bs, real, sim, 10.0, act)
    _check(disc, ws, bs, real, sim, 0.0, act)


@pytest.mark.parametrize("act", ["elu", "tanh"])
@pytest.mark.parametrize("dims,rows", [([33, 321, 40, 1], (17, 16)), ([20, 64, 330, 17, 1], (33, 40)), ([324, 32, 70, 33, 1], (3, 65))])
def test_discriminator_chain_of_launches(act, dims, rows):
    """A launch per product (a layer or the input over 320 wide): hidden chains whose second derivative counts, so that what one hidden layer's launch leaves
    for the penalty's sweep back (W^T d and d itself) reaches the next one's gradient.  Rows and widths around the 32 x 32 tiles."""
    from ksim_amd.mlp import MLP

    ws, bs = _params(dims, seed=sum(dims))
    disc = MLP(ws, bs, activation=act, dtype="f32")
    disc.train_init()
    rng = np.random.default_rng(rows[0])
    real, sim = (rng.normal(size=(n, 1, dims[0])).astype(np.float32) for n in rows)
    assert _check(disc, ws, bs, real, sim, 10.0, act)[2] > 1e-3
    _check(disc, ws, bs, real, sim, 0.0, act)


@pytest.mark.parametrize("dims,limit,coef", [([12, 32, 16, 1], 24576, 10.0), ([140, 32, 1], 8192, 0.0), ([40, 33, 1], 65536, 10.0),
                                             ([9, 64, 1], 16384, 0.0), ([9, 40, 48, 1], 65536, 0.0), ([9, 49, 20, 1], 65536, 10.0), ([9, 65, 1], 16384, 0.0)])
def test_discriminator_on_both_sides_of_the_row_limits(dims, limit, coef):
    """Narrow hidden layers change from one launch for the whole chain to a launch per product where the rows fill the chip: the last row count of the one
    and the first of the other, and the narrowest networks that never change.  Sums of up to 65537 rows in fp32 slices of a few hundred: far inside the file's tolerance."""
    from ksim_amd.mlp import MLP

    ws, bs = _params(dims, seed=sum(dims))
    disc = MLP(ws, bs, activation="elu", dtype="f32")
    disc.train_init()
    rng = np.random.default_rng(limit)
    for rows in (limit, limit + 1):
        real, sim = (rng.normal(size=(n, 1, dims[0])).astype(np.float32) for n in (rows // 3, rows - rows // 3))
        _check(disc, ws, bs, real, sim, coef, "elu")


def test_discriminator_products_are_as_precise_as_four_partial_sums():
    """A product over 256 columns in the launch for a frame's whole chain is no further from 64 bits than the launches per product, whose four wavefronts
    sum a quarter of the reduction each (here restated in numpy: fused multiply-adds in fp32, then the four sums).  With output weights of zero
    the one real frame's error is -1 and the simulated frame of zeros leaves nothing, so the output weights' gradient is minus the hidden layer, bit for bit."""
    from ksim_amd.mlp import MLP

    K, got, four = 256, [], []
    for seed in range(8):
        rng = np.random.default_rng(seed)
        w, x = (rng.normal(size=s).astype(np.float32) for s in ((K, K), K))
        disc = MLP([w, np.zeros((1, K), np.float32)], [np.zeros(K, np.float32), np.zeros(1, np.float32)], activation="relu", dtype="f32")
        disc.train_init()
        disc.disc_loss_grad(torch.tensor(x, device=DEV).reshape(1, 1, K), torch.zeros(1, 1, K, device=DEV), 0.0)
        y = -disc.parameters(gradients=True)[1][0].double().cpu().numpy().ravel()
        exact = w.astype(np.float64) @ x.astype(np.float64)
        sums = np.zeros((4, K), np.float32)
        for k in range(K // 4):
            for q in range(4):
                sums[q] = (sums[q] + w[:, q * K // 4 + k].astype(np.float64) * x[q * K // 4 + k]).astype(np.float32)
        total = ((sums[0] + sums[1]) + sums[2]) + sums[3]
        scale = np.linalg.norm(np.maximum(exact, 0))
        got.append((y - np.maximum(exact, 0)) / scale)
        four.append((np.maximum(total, 0) - np.maximum(exact, 0)) / scale)
    # 1000 entries' root mean square: its own spread is 2 %, two long sums would be 1.35 times the bound and the present ones are 0.65 of it
    assert np.linalg.norm(got) <= np.linalg.norm(four)


def test_discriminator_reduction_tail_leaves_infinite_weights_alone():
    """A reduction over 20 units is padded to 32: an infinite weight in its last row reaches the gradients as the infinity it is (every other
    factor is positive and finite), not as the NaN of an infinity times a padding zero."""
    from ksim_amd.mlp import MLP

    rng = np.random.default_rng(4)
    dims = [4, 20, 20, 1]
    ws = [rng.uniform(0.1, 1.0, size=(o, i)).astype(np.float32) for i, o in zip(dims[:-1], dims[1:])]
    bs = [np.zeros(o, dtype=np.float32) for o in dims[1:]]
    ws[1][19, 7] = np.inf
    disc = MLP(ws, bs, activation="relu", dtype="f32")
    disc.train_init()
    x = rng.uniform(0.1, 1.0, size=(1, 5, 4)).astype(np.float32)
    disc.disc_loss_grad(torch.tensor(x, device=DEV), torch.tensor(x + 1.0, device=DEV), 0.0)
    tw, tb = ([torch.tensor(p, dtype=torch.float64, requires_grad=True) for p in params] for params in (ws, bs))
    sum(0.5 * ((oup.mlp(torch.tensor(f, dtype=torch.float64), tw, tb, "relu") - t) ** 2).sum() for f, t in ((x, 1.0), (x + 1.0, -1.0))).backward()
    for (got, _), want in zip(disc.parameters(gradients=True), tw):
        assert torch.isposinf(want.grad).all()
        assert torch.isposinf(got).all()


def test_discriminator_update_learns_and_matches_oracle_steps():
    """Three optimiser steps on fixed batches against the oracle's Adam (the optax chain restated for the policy update),
    then the loop with sampled batches: the loss on separable data goes down."""
    from ksim_amd import amp
    from ksim_amd.mlp import MLP

    dims = [8, 32, 1]
    ws, bs = _params(dims, seed=21)
    disc = MLP(ws, bs, activation="elu", dtype="f32")
    cfg = amp.AMPConfig(amp_reference_batch_size=4, disc_num_passes=2, amp_grad_penalty_coef=5.0, learning_rate=1e-2, max_grad_norm=1.0)
    upd = amp.DiscriminatorUpdate(disc, cfg)
    rng = np.random.default_rng(2)
    real = (rng.normal(size=(4, 6, 8)) + 1.0).astype(np.float32)
    sim = (rng.normal(size=(4, 6, 8)) - 1.0).astype(np.float32)
    # oracle: gradient, global-norm clip, Adam with bias correction
    pw, pb = [w.astype(np.float64) for w in ws], [b.astype(np.float64) for b in bs]
    m1 = [np.zeros_like(p) for p in pw + pb]; m2 = [np.zeros_like(p) for p in pw + pb]
    for step in range(1, 4):
        upd.step(torch.tensor(real, device=DEV), torch.tensor(sim, device=DEV))
        _, g = oamp.disc_loss_and_grads(pw, pb, real, sim, cfg.amp_grad_penalty_coef, act="elu")
        flat = [gw for gw, _ in g] + [gb for _, gb in g]
        norm = np.sqrt(sum((x ** 2).sum() for x in flat))
        flat = [x * min(1.0, cfg.max_grad_norm / norm) for x in flat]
        for i, (p, x) in enumerate(zip(pw + pb, flat)):
            m1[i] = 0.9 * m1[i] + 0.1 * x
            m2[i] = 0.999 * m2[i] + 0.001 * x * x
            p -= cfg.learning_rate * (m1[i] / (1 - 0.9 ** step)) / (np.sqrt(m2[i] / (1 - 0.999 ** step)) + 1e-8)
    for (gw, gb), w, b in zip(disc.parameters(), pw, pb):
        np.testing.assert_allclose(gw.cpu().numpy(), w, rtol=0, atol=2e-4)
        np.testing.assert_allclose(gb.cpu().numpy(), b, rtol=0, atol=2e-4)
    # the network that the rollout's forward pass uses follows the master weights
    x = torch.tensor(real.reshape(-1, 8), device=DEV)
    want = oup.mlp(torch.tensor(real.reshape(-1, 8), dtype=torch.float64), [torch.tensor(w) for w in pw], [torch.tensor(b) for b in pb]).numpy()
    np.testing.assert_allclose(disc(x).cpu().numpy(), want, rtol=0, atol=1e-3)

    gen = torch.Generator().manual_seed(0)
    clips = torch.tensor((rng.normal(size=(5, 4, 8)) + 1.0).astype(np.float32), device=DEV)   # clips shorter than the window: they loop
    sims = torch.tensor((rng.normal(size=(16, 6, 8)) - 1.0).astype(np.float32), device=DEV)
    first = upd.update(clips, sims, gen)
    for _ in range(30):
        last = upd.update(clips, sims, gen)
    assert float(last["disc_loss"]) < 0.5 * float(first["disc_loss"])
    assert set(last) == {"disc_loss", "disc_real_loss", "disc_sim_loss", "disc_gp_loss"}


def test_discriminator_argument_errors():
    from ksim_amd import _lib, amp
    from ksim_amd.mlp import MLP

    ws, bs = _params([6, 8, 2], seed=1)
    two = MLP(ws, bs, activation="elu", dtype="f32")
    with pytest.raises(_lib.KsError, match="one number"):
        amp.DiscriminatorUpdate(two, amp.AMPConfig())
    ws, bs = _params([6, 8, 1], seed=1)
    gelu = MLP(ws, bs, activation="gelu", dtype="f32")
    gelu.train_init()
    x = torch.zeros(2, 3, 6, device=DEV)
    with pytest.raises(_lib.KsError, match="GELU"):
        gelu.disc_loss_grad(x, x, 1.0)
    with pytest.raises(ValueError, match="must divide"):
        amp.make_sim_batch(torch.zeros(10, 3, 6, device=DEV), 4, torch.Generator())
    w = amp.loop_slice(torch.arange(3, device=DEV), 2, 5)
    assert w.tolist() == [2, 0, 1, 2, 0]
    # a batch of reference windows is those slices, of the clips and starts the generator draws, gathered at once
    motions = torch.arange(4 * 7 * 2, device=DEV, dtype=torch.float32).reshape(4, 7, 2)
    batch = amp.make_real_batch(motions, 10, 6, torch.Generator().manual_seed(5))
    g = torch.Generator().manual_seed(5)
    clips, starts = torch.randint(0, 4, (6,), generator=g), torch.randint(0, 7, (6,), generator=g)
    want = torch.stack([amp.loop_slice(motions[int(c)], int(s0), 10) for c, s0 in zip(clips, starts)])
    assert batch.shape == (6, 10, 2) and torch.equal(batch, want)


@pytest.mark.parametrize("dims,shapes", [((5, 33, 1), ((1, 1), (2, 3))), ((71, 128, 96, 1), ((3, 11), (1, 33))), ((64, 32, 1), ((4, 8), (0, 1))),
                                         ((64, 32, 1), ((0, 1), (4, 8))), ((40, 256, 64, 1), ((2, 700), (3, 1000)))])
def test_discriminator_gradient_at_the_edges_of_its_tiles(dims, shapes):
    """Rows and widths around the 32 x 32 tiles and the 32-step chunks of the weight gradients, frames that are not 16-byte rows, either set
    of motions empty, and row counts that cut the weight gradients into slices.  fp32 against float64 autograd: sums of up to 4400
    rows, each rounded at 2^-24 of its size."""
    from ksim_amd.mlp import random_mlp

    rng = np.random.default_rng(sum(dims))
    net, ws, bs = random_mlp(dims, 3, dtype="f32")
    net.train_init()
    real, sim = (rng.normal(size=(*s, dims[0])) for s in shapes)
    losses = net.disc_loss_grad(torch.tensor(real, dtype=torch.float32, device=DEV), torch.tensor(sim, dtype=torch.float32, device=DEV), 10.0)
    tw, tb = [torch.tensor(w, dtype=torch.float64, requires_grad=True) for w in ws], [torch.tensor(b, dtype=torch.float64, requires_grad=True) for b in bs]

    def score(x):
        for i, (w, b) in enumerate(zip(tw, tb)):
            x = x @ w.T + b
            x = torch.nn.functional.elu(x) if i + 1 < len(tw) else x
        return x[..., 0]

    r, s = torch.tensor(real, requires_grad=True), torch.tensor(sim)
    out = score(r)
    terms = [0.5 * ((out - 1) ** 2).sum(), 0.5 * ((score(s) + 1) ** 2).sum(), torch.zeros((), dtype=torch.float64)]
    if real.size:
        g, = torch.autograd.grad(out.sum(), r, create_graph=True)
        terms[2] = 5.0 * (g ** 2).sum() / real.shape[0]
    sum(terms).backward()
    for got, want in zip(losses.tolist(), terms):
        assert abs(got - want.item()) <= 1e-5 * max(1.0, abs(want.item()))
    for (gw, gb), w, b in zip(net.parameters(gradients=True), tw, tb):
        for got, want in ((gw, w.grad), (gb, b.grad)):
            assert np.abs(got.cpu().numpy() - want.numpy()).max() <= 2e-5 * max(np.abs(want.numpy()).max(), 1e-3)


def test_discriminator_over_more_rows_than_a_grid_dimension_counts_tiles():
    """Two million frames and more (65536 row tiles of 32) against the same gradient added up over parts of them.  Frames repeat every 4096 rows,
    so the result is a known multiple of one period's: sums of R terms in fp32 slices, each rounding 2^-24 of a partial sum."""
    from ksim_amd.mlp import random_mlp

    period, repeats = 4096, 520  # 2 129 920 rows
    real = torch.randn(1, period, 6, device=DEV)
    grads = []
    for n in (1, repeats):
        net, _, _ = random_mlp((6, 8, 1), 3, dtype="f32")
        net.train_init()
        # penalty: the mean over motions, so that `n` motions of one period each carry the same share
        losses = net.disc_loss_grad(real.expand(n, period, 6).contiguous(), torch.empty(0, 1, 6, device=DEV), 10.0)
        grads.append((losses.double(), [g.double() for pair in net.parameters(gradients=True) for g in pair]))
    (l1, g1), (ln, gn) = grads
    assert torch.allclose(ln, torch.stack([l1[0] * repeats, l1[1], l1[2]]), rtol=1e-5)
    # the squared-error gradient grows with the repeats, the penalty's does not: take the latter from a run of its own size
    net, _, _ = random_mlp((6, 8, 1), 3, dtype="f32")
    net.train_init()
    net.disc_loss_grad(real, torch.empty(0, 1, 6, device=DEV), 0.0)
    g0 = [g.double() for pair in net.parameters(gradients=True) for g in pair]
    for a, b, c in zip(g0, g1, gn):
        want = a * repeats + (b - a)
        assert (c - want).abs().max() <= 1e-4 * want.abs().max()


def test_reference_windows_of_strided_clips_are_gathered_in_place():
    """Clips given as a slice of a larger array or expanded along an axis: the same windows, and no copy of the clips."""
    from ksim_amd import amp

    whole = torch.randn(6, 40, 3, 8, device=DEV)
    views = [whole[:, ::2, 1], whole[1::2, 5:, 2, :5], whole[:1, :, 0].expand(64, 40, 8), whole[:, :1, 0].expand(6, 4000, 8), whole[:, :, 0, 2:3]]
    for motions in views:
        want = amp.make_real_batch(motions.contiguous(), 10, 6, torch.Generator().manual_seed(5))
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        got = amp.make_real_batch(motions, 10, 6, torch.Generator().manual_seed(5))
        assert torch.equal(got, want)
        if motions.numel() > 16384:
            assert torch.cuda.max_memory_allocated() - before < motions.numel() * 4
    big = torch.zeros(1, 1, 1, device=DEV).expand(100000, 100000, 64)  # 2.5 TB if it were copied
    assert amp.make_real_batch(big, 4, 2, torch.Generator().manual_seed(1)).shape == (2, 4, 64)


@pytest.mark.parametrize("rows", [((3, 13), (2, 45)), ((7, 101), (3, 467))])
@pytest.mark.parametrize("coef", [0.0, 10.0])
def test_discriminator_of_five_layers(rows, coef):
    """One reduction over the penalty's rows and then all rows per weight gradient, every layer in one launch: row counts at which the two meet
    inside a 32-step chunk and a slice, with one slice and with several."""
    from ksim_amd.mlp import MLP

    dims = [17, 40, 33, 64, 20, 1]
    ws, bs = _params(dims, seed=9)
    disc = MLP(ws, bs, activation="tanh", dtype="f32")
    disc.train_init()
    rng = np.random.default_rng(rows[0][1])
    real, sim = (rng.normal(size=(*s, dims[0])).astype(np.float32) for s in rows)
    for _ in range(2):  # counters and partial sums of the first call do not reach the second
        _check(disc, ws, bs, real, sim, coef, "tanh")


@pytest.mark.parametrize("batch,envs,window_t,clips,clip_t,frame", [(1, 1, 1, 1, 1, 1), (6, 12, 10, 4, 7, 2), (2, 4, 40, 3, 3, 65), (32, 64, 32, 9, 50, 71),
                                                                    (128, 128, 24, 5, 24, 86), (129, 129, 8, 3, 9, 3)])
def test_both_batches_of_a_step_in_one_launch(batch, envs, window_t, clips, clip_t, frame):
    """The batches that `update` draws are those of `make_real_batch` and `make_sim_batch` from the same generator: windows that wrap once and
    several times, the largest batch of the launch and one more than it takes, and arrays that it leaves to them."""
    from ksim_amd import amp

    g = torch.Generator(device=DEV).manual_seed(batch)
    motions, sims = torch.randn(clips, clip_t, frame, device=DEV, generator=g), torch.randn(envs, window_t, frame, device=DEV, generator=g)
    strided = torch.randn(clips, 2 * clip_t, frame, device=DEV, generator=g)[:, ::2]
    for m, s in ((motions, sims), (strided, sims), (motions.double(), sims.double()), (motions, sims.expand(envs, window_t, frame))):
        one, two = torch.Generator().manual_seed(7), torch.Generator().manual_seed(7)
        real, sim = amp._batches(m, s, batch, one)
        assert torch.equal(real, amp.make_real_batch(m, window_t, batch, two)) and torch.equal(sim, amp.make_sim_batch(s, batch, two))
        assert torch.equal(one.get_state(), two.get_state())
    with pytest.raises(ValueError, match="must divide"):
        amp._batches(motions, torch.cat([sims, sims[:1]]) if batch > 1 else sims, 2 if batch == 1 else batch, torch.Generator())


@pytest.mark.parametrize("device", ["meta", "cuda"])
def test_indices_drawn_off_the_host_are_not_read_there(device, monkeypatch):
    """Under a default device the draws are not host memory, which is where the launcher of both batches reads them: such a call goes to the
    functions of the single batches, which refuse it."""
    from ksim_amd import _lib, amp

    class Library:
        def __getattr__(self, name):
            raise AssertionError(name)

    motions, sims = torch.randn(3, 7, 5, device=DEV), torch.randn(4, 6, 5, device=DEV)
    monkeypatch.setattr(_lib, "load", lambda: Library())
    generator = torch.Generator(device="cpu" if device == "meta" else DEV)
    with torch.device(device), pytest.raises(RuntimeError):
        amp._batches(motions, sims, 2, generator)


def test_batches_drawn_under_capture_are_left_to_the_functions_that_refuse_them(monkeypatch):
    """A graph that held a step's draws would replay them for ever; the upload of the drawn indices is what no capture takes."""
    from ksim_amd import amp

    def windows(*args):
        raise NotImplementedError("left to the single batches")

    motions, sims = torch.randn(3, 7, 5, device=DEV), torch.randn(4, 6, 5, device=DEV)
    monkeypatch.setattr(amp, "_windows", windows)
    with pytest.raises(NotImplementedError), torch.cuda.graph(torch.cuda.CUDAGraph()):
        sims + 1.0
        amp._batches(motions, sims, 2, torch.Generator())
    monkeypatch.undo()
    real, sim = amp._batches(motions, sims, 2, torch.Generator())
    assert real.shape == sim.shape == (2, 6, 5)


@pytest.mark.parametrize("window_t", [134214, 134215, 134216])
def test_windows_at_the_launch_limit(window_t):
    """The longest windows that the launch takes, and those that it leaves to the functions of the single batches: 1000 floats a frame, a clip of one
    frame, at most 65535 blocks of 2048 floats of clip and window."""
    from ksim_amd import amp

    motions, sims = torch.randn(1, 1, 1000, device=DEV), torch.randn(1, window_t, 1000, device=DEV)
    one, two = torch.Generator().manual_seed(7), torch.Generator().manual_seed(7)
    real, sim = amp._batches(motions, sims, 1, one)
    assert torch.equal(real, amp.make_real_batch(motions, window_t, 1, two)) and torch.equal(sim, amp.make_sim_batch(sims, 1, two))
