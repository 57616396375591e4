"""MLP forward on the matrix cores against a float64 torch reference (F.linear + F.elu)."""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def reference(x, ws, bs, act, bf16):
    """float64 library reference; for the bf16 path weights and layer inputs are rounded to bf16 first."""
    rnd = (lambda t: t.to(torch.bfloat16).to(torch.float64)) if bf16 else (lambda t: t.to(torch.float64))
    h = torch.from_numpy(x)
    fn = {"elu": F.elu, "relu": F.relu, "tanh": torch.tanh, None: lambda t: t, "none": lambda t: t}[act]
    for i, (w, b) in enumerate(zip(ws, bs)):
        h = F.linear(rnd(h.to(torch.float32)), rnd(torch.from_numpy(w)), torch.from_numpy(b).to(torch.float64))
        if i + 1 < len(ws):
            h = fn(h)
    return h.numpy()


@pytest.mark.parametrize("dims,dtype,act,M", [
    ((71, 256, 256, 256, 21), "f32", "elu", 300),      # benchmark config 3 actor
    ((68, 512, 512, 512, 20), "bf16", "elu", 1000),    # config 4 actor
    ((68, 512, 512, 512, 1), "bf16", "elu", 129),      # config 4 critic, ragged tile
    ((71, 256, 256, 1), "bf16", "relu", 64),           # config 5 discriminator shape
    ((5, 3), "f32", None, 7), ((40, 100, 9), "f32", "tanh", 1), ((33, 130, 130, 2), "bf16", "tanh", 257),
    ((68, 512, 512, 512, 20), "bf16", "elu", 16384 + 45),   # 64-row tiles of the whole-network kernel
    ((68, 512, 512, 512, 20), "bf16", "elu", 32768 + 77),   # 128-row tiles
    ((71, 256, 256, 1), "bf16", "relu", 40000),             # 128-row tiles, one output tile per wavefront
    ((64, 1024, 8), "bf16", "elu", 500),                    # wider than the whole-network kernel takes: per-layer path
    ((600, 64, 3), "bf16", "none", 100),
])
def test_mlp_matches_reference(dims, dtype, act, M):
    from ksim_amd.mlp import MLP

    rng = np.random.default_rng(sum(dims) + M)
    ws = [rng.normal(scale=1 / np.sqrt(i), size=(o, i)).astype(np.float32) for i, o in zip(dims[:-1], dims[1:])]
    bs = [rng.normal(scale=0.1, size=o).astype(np.float32) for o in dims[1:]]
    x = rng.normal(size=(M, dims[0])).astype(np.float32)
    net = MLP(ws, bs, activation=act if act not in (None, "none") else "none", dtype=dtype)
    y = net(torch.from_numpy(x).to(DEV)).cpu().numpy()
    want = reference(x, ws, bs, act, dtype == "bf16")
    scale = np.abs(want).max()
    # f32: fp32 accumulation error only; bf16: inputs rounded identically, so only accumulation order differs,
    # plus re-rounding of hidden activations that land on a bf16 tie
    tol = 2e-5 if dtype == "f32" else 6e-3
    assert np.abs(y - want).max() <= tol * scale, np.abs(y - want).max() / scale
    assert net.flops_per_row() == 2 * sum(a * b for a, b in zip(dims[:-1], dims[1:]))


def test_mlp_rows_are_independent_and_errors():
    from ksim_amd import _lib
    from ksim_amd.mlp import random_mlp

    net, ws, bs = random_mlp((68, 512, 512, 512, 20), seed=3)
    x = torch.randn(700, 68, device=DEV)
    y = net(x)
    y2 = net(x[123:460].contiguous())
    assert torch.equal(y[123:460], y2)
    big = torch.randn(33000, 68, device=DEV)  # another row tile size, same bits per row
    assert torch.equal(net(big)[5000:5700], net(big[5000:5700].contiguous()))
    with pytest.raises(_lib.KsError):
        net(torch.randn(4, 67, device=DEV))
    with pytest.raises(_lib.KsError):
        net(torch.randn(4, 68))
    assert net(torch.empty(0, 68, device=DEV)).shape == (0, 20)


@pytest.mark.parametrize("M", [8192, 777, 20000])
def test_paired_forward_equals_two_single_forwards(M):
    """Actor and critic over the same rows in one launch (below 16384 rows) or two: bit-identical to separate calls,
    also for networks of different widths and for a pair that cannot share a launch."""
    from ksim_amd import _lib
    from ksim_amd.mlp import random_mlp

    actor, _, _ = random_mlp((68, 512, 512, 512, 20), seed=5)
    critic, _, _ = random_mlp((68, 512, 512, 512, 1), seed=6)
    narrow, _, _ = random_mlp((68, 256, 256, 1), seed=7)
    wide, _, _ = random_mlp((68, 1024, 1), seed=8)  # per-layer path: the pair falls back to two launches
    x0, x1 = torch.randn(M, 68, device=DEV), torch.randn(M, 68, device=DEV)
    for other in (critic, narrow, wide):
        y0 = torch.full((M, 20), 7.0, device=DEV)
        y1 = torch.full((M, 1), 7.0, device=DEV)
        actor.forward_pair(x0, y0, other, x1, y1)
        assert torch.equal(y0, actor(x0)) and torch.equal(y1, other(x1))
    with pytest.raises(_lib.KsError):
        actor.forward_pair(x0, torch.empty(M, 20, device=DEV), critic, x1[:-1], torch.empty(M - 1, 1, device=DEV))


@pytest.mark.parametrize("dims", [
    (68, 512, 512, 512, 20),      # output tile cut over four wavefronts
    (71, 256, 256, 256, 33),      # two output tiles, two wavefronts each; rows of the input on no 16-byte boundary
    (5, 40, 3), (33, 130, 130, 2),
    (128, 512), (97, 140), (475, 128), (40, 1),  # single layers: 1024 tiles are the last batch of the kernel for few rows
])
def test_fp32_batches_of_every_size_give_a_row_the_same_bits(dims):
    """Few rows (32 x 32 tiles, a launch per layer), 32-row and 64-row whole-network tiles, per-layer tiles of 64 and 128 rows: the last row
    count of one kernel and the first of the next, ragged ends included."""
    from ksim_amd.mlp import MLP

    rng = np.random.default_rng(sum(dims))
    ws = [rng.normal(scale=1 / np.sqrt(i), size=(o, i)).astype(np.float32) for i, o in zip(dims[:-1], dims[1:])]
    bs = [rng.normal(scale=0.1, size=o).astype(np.float32) for o in dims[1:]]
    net = MLP(ws, bs, activation="elu", dtype="f32")
    sizes = {1, 31, 33, 65, 4000, 16383, 16384 + 37}
    if len(dims) == 2:
        few, wide = 1024 // ((dims[1] + 31) // 32) * 32, 400 // ((dims[1] + 127) // 128) * 128
        sizes |= {few, few + 1, wide - 128, wide + 37}
    else:
        sizes |= {2048, 2049}
    sizes = sorted(sizes)
    x = rng.normal(size=(max(sizes), dims[0])).astype(np.float32)
    X = torch.from_numpy(x).to(DEV)
    want = reference(x, ws, bs, "elu", False)
    full = net(X)
    # a rounding of 2^-24 per product and sum, of sums of at most 512 terms whose squares add up to about 1, over at most 4 layers
    assert np.abs(full.cpu().numpy() - want).max() <= 2e-5 * np.abs(want).max()
    for M in sizes:
        assert torch.equal(net(X[:M].contiguous()), full[:M]), M
        y0, y1 = torch.full((M, dims[-1]), 7.0, device=DEV), torch.full((M, dims[-1]), 7.0, device=DEV)
        other = MLP(ws, bs, activation="elu", dtype="f32")
        net.forward_pair(X[:M].contiguous(), y0, other, X[-M:].contiguous(), y1)
        assert torch.equal(y0, full[:M]) and torch.equal(y1, full[-M:]), M


@pytest.mark.parametrize("M", [1, 33, 4000, 20000])
def test_single_fp32_layers_keep_the_range_of_fp32(M):
    """Single layers multiply operands cut into bf16 parts: values near the largest float, tiny ones, infinities, NaN and products that
    overflow come out as the fp32 product has them."""
    from ksim_amd.mlp import MLP

    values = np.array([3.4028235e38, -3.4028235e38, 3.3961776e38, 2.0 ** -100, 1 + 2.0 ** -23, np.inf, -np.inf, np.nan, 0.1], np.float32)
    weights = np.array([1.0, -1.0, 301.3, -0.0013, 1.0 + 2.0 ** -20], np.float32)
    w = np.zeros((200, 20), np.float32)
    w[:, 3] = np.resize(weights, 200)
    x = np.zeros((M, 20), np.float32)
    x[:, 3] = np.resize(values, M)
    y = MLP([w], [np.zeros(200, np.float32)], activation="none", dtype="f32")(torch.from_numpy(x).to(DEV)).cpu().numpy()
    with np.errstate(over="ignore", invalid="ignore"):
        want = x[:, 3:4] * w[:, 3][None, :]
    assert np.array_equal(np.isnan(y), np.isnan(want)) and np.array_equal(np.isinf(y), np.isinf(want))
    finite = np.isfinite(want)
    assert np.array_equal(y[~finite & ~np.isnan(want)], want[~finite & ~np.isnan(want)])
    # eight products of 16 significant bits each are exact, the one left out is below 2^-32; the sum of the seven small ones, below 2^-6 of the
    # result, rounds six times and the last sum once, as does the product it is compared with
    assert np.all(np.abs(y[finite] - want[finite]) <= 2.0 ** -22.9 * np.abs(want[finite]))


@pytest.mark.parametrize("M", [1, 33, 4000, 20000])
def test_tiny_values_in_single_fp32_layers(M):
    """Values whose second and third bf16 parts are denormal or below the smallest: each part rounds by at most 2^-134 (bf16 ends at 2^-133), so a
    product is off by 2^-133 of the other operand, beside its own roundings."""
    from ksim_amd.mlp import MLP

    rng = np.random.default_rng(M)
    tiny = np.ldexp(rng.uniform(1, 2, 4096), rng.integers(-126, -98, 4096)).astype(np.float32) * rng.choice([-1.0, 1.0], 4096).astype(np.float32)
    plain = rng.uniform(1, 2, 4096).astype(np.float32)
    for xv, wv in ((tiny, plain), (plain, tiny)):
        x, w = np.zeros((M, 20), np.float32), np.zeros((200, 20), np.float32)
        x[:, 3], w[:, 3] = np.resize(xv, M), wv[:200]
        y = MLP([w], [np.zeros(200, np.float32)], activation="none", dtype="f32")(torch.from_numpy(x).to(DEV)).cpu().numpy().astype(np.float64)
        want = x[:, 3:4].astype(np.float64) * w[:, 3].astype(np.float64)[None, :]
        assert np.all(np.abs(y - want) <= 2.0 * 2.0 ** -133 + 2.0 ** -23.9 * np.abs(want) + 2.0 ** -149)


@pytest.mark.parametrize("dims", [(128, 384), (340, 128), (97, 70), (128, 510), (33, 5)])
def test_single_bf16_layers_of_every_batch_size(dims):
    """32-, 64- and 128-row tiles of a single bf16 layer, with a lane per feature or (narrow layers) per row: the first and last row count
    of each, ragged ends, the same bits for a row in all of them, nothing written past the output."""
    from ksim_amd.mlp import MLP

    rng = np.random.default_rng(sum(dims))
    w = (rng.normal(size=(dims[1], dims[0])) / np.sqrt(dims[0])).astype(np.float32)
    b = rng.normal(scale=0.1, size=dims[1]).astype(np.float32)
    net = MLP([w], [b], activation="none", dtype="bf16")
    sizes = [1, 31, 33, 16383, 16384 + 37, 32767, 32768 + 45]
    x = rng.normal(size=(max(sizes), dims[0])).astype(np.float32)
    X = torch.from_numpy(x).to(DEV)
    full = net(X)
    want = reference(x, [w], [b], "none", True)
    # products of bf16 values are exact in fp32: a rounding of 2^-24 per sum of up to 340 terms whose squares add up to about 1
    assert np.abs(full.cpu().numpy() - want).max() <= 2e-5 * np.abs(want).max()
    for M in sizes:
        y = torch.full((M * dims[1] + 64,), 7.0, device=DEV)
        got = net(X[:M].contiguous(), out=y[:M * dims[1]].view(M, dims[1]))
        assert torch.equal(got, full[:M]) and torch.equal(y[M * dims[1]:], torch.full((64,), 7.0, device=DEV)), M


@pytest.mark.parametrize("dims,dtype", [((68, 512, 512, 20), "f32"), ((30, 320, 5), "f32"), ((30, 256, 5), "f32"), ((68, 640, 20), "f32"),
                                        ((128, 512), "f32"), ((68, 512, 512, 20), "bf16"), ((128, 384), "bf16"), ((68, 640, 20), "bf16")])
def test_scratch_for_the_largest_batch_does_for_smaller_ones(dims, dtype):
    """A caller sizes one buffer for its largest batch: none of the size queries may shrink as the row count grows, and a small batch given
    that buffer writes nothing behind it."""
    from ksim_amd import _lib
    from ksim_amd.mlp import random_mlp

    net, _, _ = random_mlp(dims, seed=sum(dims), dtype=dtype)
    rows = sorted({0, 1, 31, 32, 33, 191, 192, 193, 256, 400, 2047, 2048, 2049, 4000, 8192, 16384, 32767, 32768, 32769, 65536, 100000, 131072})
    lib, handle = _lib.load(), net._handle
    for size in (lambda M: lib.ks_mlp_workspace_bytes(handle, M), lambda M: lib.ks_mlp_train_workspace_bytes(handle, M),
                 lambda M: lib.ks_mlp_disc_workspace_bytes(handle, M, 2 * M)):
        need = [int(size(M)) for M in rows]
        assert need == sorted(need), list(zip(rows, need))
    need, M = int(lib.ks_mlp_workspace_bytes(handle, 5000)), 256
    buf = torch.full((need + 4096,), 0x5A, dtype=torch.uint8, device=DEV)
    x, y = torch.randn(M, dims[0], device=DEV), torch.empty(M, dims[-1], device=DEV)
    _lib.check(lib.ks_mlp_forward(handle, _lib.current_stream(), M, _lib.ptr(x), _lib.ptr(y), _lib.ptr(buf)))
    assert torch.equal(buf[need:], torch.full((4096,), 0x5A, dtype=torch.uint8, device=DEV))
    assert torch.equal(y, net(x))


def _error_in_roundings(got, want):
    """Largest and root mean square relative error in units of 2^-24, one rounding of fp32."""
    e = np.abs(got.astype(np.float64) - want) / np.abs(want) * 2.0 ** 24
    return e.max(), np.sqrt((e ** 2).mean())


@pytest.mark.parametrize("M", [1, 33, 4000, 20000])
def test_single_products_of_fp32_layers_round_once(M):
    """Reductions of one term: forward (one input), input gradient (one output) and weight gradient (one row), and one term among zeros.  The
    operands' parts are exact, eight of their nine products are added and the ninth is 2^-32, so what rounds is the final sum: 1 unit at most and
    0.42 root mean square for uniformly spread results, plus seven roundings of the small products' sum, 2^-6 of it each."""
    from ksim_amd.mlp import MLP

    rng = np.random.default_rng(M)
    u = lambda *s: (rng.uniform(1, 2, s) * rng.choice([-1.0, 1.0], s)).astype(np.float32)  # noqa: E731
    n = 130
    x, w, b0 = u(M, 1), u(n, 1), np.zeros(n, np.float32)
    cases = {}
    cases["forward"] = (MLP([w], [b0], activation="none", dtype="f32")(torch.from_numpy(x).to(DEV)), x.astype(np.float64) * w[:, 0].astype(np.float64))
    rows = np.zeros((M, 40), np.float32)
    at = rng.integers(0, 40, M)
    rows[np.arange(M), at] = x[:, 0]
    wide = u(n, 40)
    cases["one input of many"] = (MLP([wide], [b0], activation="none", dtype="f32")(torch.from_numpy(rows).to(DEV)),
                                  x.astype(np.float64) * wide.T.astype(np.float64)[at])
    critic = u(1, n)
    net = MLP([critic], [np.zeros(1, np.float32)], activation="none", dtype="f32")
    net.train_init()
    inputs, dx = torch.from_numpy(u(M, n)).to(DEV), torch.empty(M, n, device=DEV)
    net.train_forward(inputs)
    net.backward_dx(inputs, torch.from_numpy(x).to(DEV), dx)
    cases["input gradient"] = (dx, x.astype(np.float64) * critic.astype(np.float64))
    net = MLP([u(70, n)], [np.zeros(70, np.float32)], activation="none", dtype="f32")
    net.train_init()
    row, dy = np.zeros((M, n), np.float32), np.zeros((M, 70), np.float32)
    row[M // 2], dy[M // 2] = u(n), u(70)
    rd, dyd = torch.from_numpy(row).to(DEV), torch.from_numpy(dy).to(DEV)
    net.train_forward(rd)
    net.backward(rd, dyd)
    cases["weight gradient"] = (net.parameters(gradients=True)[0][0], np.outer(dy[M // 2].astype(np.float64), row[M // 2].astype(np.float64)))
    for name, (got, want) in cases.items():
        worst, rms = _error_in_roundings(got.cpu().numpy(), want)
        assert worst <= 1.15 and (rms <= 0.45 or want.size < 1000), (name, worst, rms)


@pytest.mark.parametrize("dims,act", [((68, 200, 100, 20), "elu"), ((40, 64, 64, 1), "tanh"), ((30, 300, 5), "relu"), ((68, 512, 320, 20), "elu"),
                                      ((68, 256, 256, 20), "gelu"), ((33, 500, 7), "gelu"), ((71, 256, 256, 21), "elu"), ((30, 640, 5), "elu"),
                                      ((128, 384), "none"), ((20, 1), "none")])
def test_fp32_training_and_inference_forward_are_bit_equal(dims, act):
    """The first ratio of a policy update is exactly one: `train_forward` and the call give a row the same bits, whatever the hidden widths
    (multiples of 32, of 128, neither), the activation and the batch; the padding the backward pass reads is zero, so its gradients are finite and
    match float64."""
    from ksim_amd.mlp import MLP

    rng = np.random.default_rng(sum(dims))
    ws = [rng.normal(scale=1 / np.sqrt(i), size=(o, i)).astype(np.float32) for i, o in zip(dims[:-1], dims[1:])]
    bs = [rng.normal(scale=0.1, size=o).astype(np.float32) for o in dims[1:]]
    net = MLP(ws, bs, activation=act, dtype="f32")
    net.train_init()
    for M in (1, 45, 2048, 2049, 16384 + 37):
        x = torch.from_numpy(rng.normal(size=(M, dims[0])).astype(np.float32)).to(DEV)
        net._tws = torch.full((int(net._lib.ks_mlp_train_workspace_bytes(net._handle, M)),), 0xFF, dtype=torch.uint8, device=DEV)  # NaN
        got = net.train_forward(x)
        assert torch.equal(got, net(x)), M
        other, y0, y1 = MLP(ws, bs, activation=act, dtype="f32"), torch.empty_like(got), torch.empty_like(got)
        net.forward_pair(x, y0, other, x, y1)
        assert torch.equal(y0, got) and torch.equal(y1, got), M
        dy = torch.from_numpy(rng.normal(size=(M, dims[-1])).astype(np.float32)).to(DEV)
        net.backward(x, dy)
        tw = [torch.tensor(w, dtype=torch.float64, requires_grad=True) for w in ws]
        h = x.double().cpu()
        fn = {"elu": F.elu, "tanh": torch.tanh, "relu": F.relu, "none": lambda t: t, "gelu": lambda t: F.gelu(t, approximate="tanh")}[act]
        for i, (w, b) in enumerate(zip(tw, bs)):
            h = F.linear(h, w, torch.from_numpy(b).double())
            h = fn(h) if i + 1 < len(tw) else h
        h.backward(dy.double().cpu())
        for (gw, _), w in zip(net.parameters(gradients=True), tw):
            # fp32 sums of up to M rows of terms whose own error is a few 2^-24; ReLU's kink is met by no row here that a rounding moves
            assert (gw.double().cpu() - w.grad).abs().max() <= 1e-4 * w.grad.abs().max()


@pytest.mark.parametrize("dims,act", [((68, 512, 512, 512, 20), "elu"), ((475, 500, 512, 33), "tanh"), ((1, 361, 384, 353, 512, 1), "relu"),
                                      ((96, 384, 400, 64), "elu"), ((97, 512, 353, 5), "gelu")])
def test_few_rows_of_wide_bf16_networks(dims, act):
    """Up to 256 rows of a wide bf16 network spread every layer over CUs, a launch per layer: the same sums in the same order as the
    whole-network kernel's, which a call without scratch takes.  Scratch is garbage at first, and misaligned once."""
    import ctypes

    from ksim_amd import _lib
    from ksim_amd.mlp import MLP

    rng = np.random.default_rng(sum(dims))
    nets = [MLP([rng.normal(scale=1 / np.sqrt(i), size=(o, i)).astype(np.float32) for i, o in zip(d[:-1], d[1:])],
                [rng.normal(scale=0.1, size=o).astype(np.float32) for o in d[1:]], activation=act, dtype="bf16")
            for d in (dims, dims[:-2] + (512, 1))]
    lib, p = nets[0]._lib, lambda t: ctypes.c_void_p(t.data_ptr())
    for M in (1, 31, 32, 33, 255, 256, 257):
        need = [lib.ks_mlp_workspace_bytes(n._handle, M) for n in nets]
        assert min(need) > 0
        ws = [torch.full((k + 8,), 255, dtype=torch.uint8, device=DEV) for k in need]
        x = [torch.randn(M, dims[0], device=DEV) for _ in nets]
        plain = [torch.empty(M, n.out_dim, device=DEV) for n in nets]
        for n, a, o in zip(nets, x, plain):
            assert lib.ks_mlp_forward(n._handle, _lib.current_stream(), M, p(a), p(o), None) == 0
        for at in (0, 4):
            out = [torch.full((M + 1, n.out_dim), 7.0, device=DEV) for n in nets]
            for n, a, o, w in zip(nets, x, out, ws):
                assert lib.ks_mlp_forward(n._handle, _lib.current_stream(), M, p(a), p(o), ctypes.c_void_p(w.data_ptr() + at)) == 0
            pair = [torch.full((M + 1, n.out_dim), 7.0, device=DEV) for n in nets]
            assert lib.ks_mlp_forward_pair(nets[0]._handle, nets[1]._handle, _lib.current_stream(), M, p(x[0]), p(pair[0]), p(x[1]), p(pair[1]),
                                           p(ws[0]), p(ws[1])) == 0
            for o, q, want in zip(out, pair, plain):
                assert torch.equal(o[:M], want) and torch.equal(q[:M], want)
                assert bool((o[M] == 7.0).all()) and bool((q[M] == 7.0).all())  # nothing behind the last row


def test_networks_optimised_together_match_one_by_one():
    """One squared norm and one optimiser step over many networks: mixed precisions, more layers than a launch's table holds, ragged widths, a
    frozen bias and a network named twice (two steps); against the same calls network by network."""
    import ctypes

    from ksim_amd import _lib, _lib_terms as T, mlp
    from ksim_amd.mlp import MLP

    shapes = [((68, 512, 512, 512, 20), "bf16"), ((33, 130, 7), "bf16"), ((128, 384), "bf16"), ((475, 128), "f32"), ((5, 3), "f32"),
              ((20, 40, 30, 20, 30, 40, 20, 10, 5), "f32"), ((9, 8, 7, 6, 5, 4, 3, 2, 1), "f32"), ((17, 70, 90, 5), "f32"), ((40, 33), "f32")]

    def make():
        rng = np.random.default_rng(5)
        nets = []
        for dims, dtype in shapes:
            net = MLP([rng.normal(scale=1 / np.sqrt(i), size=(o, i)).astype(np.float32) for i, o in zip(dims[:-1], dims[1:])],
                      [rng.normal(scale=0.1, size=o).astype(np.float32) for o in dims[1:]], activation="elu", dtype=dtype)
            net.train_init()
            x = torch.from_numpy(rng.normal(size=(96, dims[0])).astype(np.float32)).to(DEV)
            net.train_forward(x)
            net.backward(x, torch.from_numpy(rng.normal(size=(96, dims[-1])).astype(np.float32)).to(DEV))
            nets.append((net, x))
        _lib.check(nets[2][0]._lib.ks_mlp_freeze_bias_prefix(nets[2][0]._handle, 0, 100))
        return nets

    one, all_ = make(), make()
    params = T.KsAdamParams(1e-2, 0.9, 0.999, 1e-8, 0.01, 0.5, 3)
    a, b = (torch.full((1,), 0.25, dtype=torch.float64, device=DEV) for _ in range(2))
    for net, _ in one:
        net.grad_sqnorm(a)
    mlp.grad_sqnorm([n for n, _ in all_], b)
    want = 0.25
    for k, (net, _) in enumerate(all_):
        for w, g in net.parameters(gradients=True):
            want += float(w.double().square().sum()) + float(g.double()[100 if k == 2 else 0:].square().sum())
    assert torch.equal(a, b) and abs(float(b) - want) < 1e-9 * want
    order = list(range(len(one))) + [1]
    for k in order:
        one[k][0].adam_step(params, a)
    mlp.adam_step([all_[k][0] for k in order], params, b)
    for (n1, x), (n2, _) in zip(one, all_):
        for (w1, b1), (w2, b2) in zip(n1.parameters(), n2.parameters()):
            assert torch.equal(w1, w2) and torch.equal(b1, b2)
        y = n2(x)  # the copies that the forward and backward passes read follow the master weights
        assert torch.equal(n1(x), y)
        ws, bs = zip(*n2.parameters())
        ref = reference(x.cpu().numpy(), [w.cpu().numpy() for w in ws], [c.cpu().numpy() for c in bs], "elu", n2.dtype == "bf16")
        assert np.abs(y.cpu().numpy() - ref).max() <= (6e-3 if n2.dtype == "bf16" else 2e-5) * np.abs(ref).max()
        dx1, dx2 = torch.empty_like(x), torch.empty_like(x)
        dy = torch.ones(x.shape[0], n2.out_dim, device=DEV)
        n1.train_forward(x); n2.train_forward(x)
        assert torch.equal(n1.backward_dx(x, dy, dx1), n2.backward_dx(x, dy, dx2))


def test_parameters_of_several_networks_in_one_launch():
    """More layers than one launch's table holds, ragged widths, weights and gradients; against the copies network by network."""
    from ksim_amd import _lib, mlp
    from ksim_amd.mlp import MLP

    rng = np.random.default_rng(6)
    nets = []
    for dims in ((33, 130, 7), (5, 3), (20, 40, 30, 20, 30, 40, 20, 10, 5), (9, 8, 7, 6, 5, 4, 3, 2, 1), (17, 257, 1)):
        net = MLP([rng.normal(size=(o, i)).astype(np.float32) for i, o in zip(dims[:-1], dims[1:])],
                  [rng.normal(size=o).astype(np.float32) for o in dims[1:]], activation="elu", dtype="f32")
        net.train_init()
        x = torch.from_numpy(rng.normal(size=(32, dims[0])).astype(np.float32)).to(DEV)
        net.train_forward(x)
        net.backward(x, torch.ones((32, dims[-1]), device=DEV))
        nets.append(net)
    for gradients in (False, True):
        for net, got in zip(nets, mlp.copy_parameters(nets, gradients)):
            want = net.parameters(gradients)
            assert len(got) == len(want) == len(net.dims) - 1
            assert all(torch.equal(a, c) and torch.equal(b, d) for (a, b), (c, d) in zip(got, want))
    assert mlp.copy_parameters([]) == []
    with pytest.raises(_lib.KsError):  # a network without a training state, behind one that has it
        mlp.copy_parameters([nets[0], MLP([np.ones((2, 3), np.float32)], [np.ones(2, np.float32)], activation="elu", dtype="f32")])


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
def test_one_network_called_by_two_threads(dtype):
    """Two threads on one stream, whose launches may alternate, and two on streams of their own: every call's rows are its own."""
    import threading

    from ksim_amd.mlp import random_mlp

    net, _, _ = random_mlp((68, 512, 512, 512, 20), seed=5, dtype=dtype)
    xs = [[torch.from_numpy(np.random.default_rng(10 * k + i).normal(size=(1 + 13 * i, 68)).astype(np.float32)).to(DEV) for i in range(5)] for k in range(2)]
    want = [[net(x) for x in rows] for rows in xs]
    shared = torch.cuda.Stream()
    for streams in ([shared, shared], [torch.cuda.Stream(), torch.cuda.Stream()]):
        got, errors = [None, None], []
        torch.cuda.synchronize()

        def work(k):
            try:
                with torch.cuda.stream(streams[k]):
                    got[k] = [[net(x) for x in xs[k]] for _ in range(20)]
            except Exception as e:  # shown by the assertion below
                errors.append(e)

        threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join(60)
        torch.cuda.synchronize()
        assert not errors and not any(t.is_alive() for t in threads)
        for k in range(2):
            for rep in got[k]:
                assert all(torch.equal(a, b) for a, b in zip(rep, want[k]))


@pytest.mark.parametrize("M", [1, 37, 193, 1544, 16411, 32771])
def test_single_layers_in_shared_launches_match_one_by_one(M):
    """Backward passes of single layers of both precisions in one call (more of them than a launch takes, odd widths, inputs that are columns
    of wider rows, without input or without weight gradient) and pairs of forward passes, bit for bit the calls by themselves."""
    from ksim_amd.mlp import MLP
    from ksim_amd.recurrent import LayerBackward, LayerForward, run_layers, run_layers_backward

    rng = np.random.default_rng(M)
    t = lambda *s: torch.from_numpy(rng.normal(size=s).astype(np.float32)).cuda()  # noqa: E731
    shapes = [(43, 128), (128, 384), (128, 384), (128, 510), (340, 128), (128, 1), (128, 40)]
    nets = []
    for dtype in ("bf16", "f32"):
        for k, (i, o) in enumerate(shapes * (2 if dtype == "bf16" and M < 2000 else 1)):  # two layers of a shape: two launches of weight gradients
            net = MLP([rng.normal(scale=i ** -0.5, size=(o, i))], [0.1 * rng.normal(size=o)], activation="none", dtype=dtype)
            net.train_init()
            nets.append((net, k))
    calls, want = [], []
    for net, k in nets:
        i, o = net.in_dim, net.out_dim
        wide = t(M, i + 32)
        x, dy = (wide[:, 32:] if k % 3 == 0 else t(M, i)), t(M, o)
        dx = torch.empty(M, i, device="cuda") if k % 4 != 3 else None
        w = k % 5 != 4 or dx is None
        if w:
            net.layer_weight_grad(x, dy)
        grads = [g.clone() for pair in net.parameters(gradients=True) for g in pair]
        one = None if dx is None else net.backward_dx(None, dy, torch.empty_like(dx), weight_gradients=False)
        net.layer_weight_grad(t(M, i), t(M, o))  # something else in the handle
        other = [g.clone() for pair in net.parameters(gradients=True) for g in pair]
        calls.append(LayerBackward(net, dy, x if w else None, dx))
        want.append((grads if w else other, one))
    run_layers_backward(calls)
    for (net, k), call, (grads, one) in zip(nets, calls, want):
        got = [g for pair in net.parameters(gradients=True) for g in pair]
        assert all(torch.equal(a, b) for a, b in zip(got, grads)), (net.dims, net.dtype)
        assert one is None or torch.equal(call.dx, one), (net.dims, net.dtype)
    forward = [LayerForward(net, t(M, net.in_dim)) for net, _ in nets]
    run_layers(forward)
    for call in forward:
        assert torch.equal(call.out, call.net(call.x)), (call.net.dims, call.net.dtype)


@pytest.mark.parametrize("hidden,dtype,act,M", [(256, "bf16", "elu", 1), (256, "bf16", "elu", 64), (256, "f32", "tanh", 37), (128, "bf16", "relu", 4099), (512, "bf16", "elu", 64),
                                                (512, "f32", "elu", 45), (256, "f32", "elu", 2500), (64, "bf16", "elu", 16383), (64, "bf16", "elu", 16390)])
def test_actions_sampled_in_the_networks_launch_match_the_launch_of_their_own(hidden, dtype, act, M):
    """Actor, critic and actions in one call against `forward_pair` and `sample_action`, bit for bit: every form of the pair's launch (the last
    rows of a tile, few rows of a wide network, rows beyond the pair's limit), drawn, given and no noise, a step counted on the device,
    means that are clipped or not a number."""
    from ksim_amd.env_terms import action_sample, sample_action
    from ksim_amd.mlp import MLP

    rng = np.random.default_rng(M)
    nets = []
    for out in (20, 1):
        dims = (68, hidden, hidden, hidden, out)
        nets.append(MLP([rng.normal(scale=i ** -0.5, size=(o, i)) for i, o in zip(dims[:-1], dims[1:])], [0.1 * rng.normal(size=o) for o in dims[1:]],
                        activation=act, dtype=dtype))
    actor, critic = nets
    t = lambda *s: torch.from_numpy(rng.normal(size=s).astype(np.float32)).cuda()  # noqa: E731
    xa, xc, log_std, noise, base = t(M, 68), t(M, 68), t(20), t(M, 20), torch.tensor([5], dtype=torch.int64, device="cuda")
    xa[M // 2, 3] = float("nan")
    for given in (dict(log_std=log_std, seed=11, step=3), dict(log_std=log_std, seed=11, step=3, step_base=base), dict(log_std=log_std, noise=noise), dict(log_std=None)):
        got, want = [[torch.full(s, 7.0, device="cuda") for s in ((M, 20), (M, 1), (M, 20))] for _ in range(2)]
        actor.forward_pair(xa, want[0], critic, xc, want[1])
        sample_action(want[0], clip_max=0.75, out=want[2], **given)
        actor.forward_pair(xa, got[0], critic, xc, got[1], action_sample(got[0], clip_max=0.75, out=got[2], **given))
        for g, w in zip(got, want):
            assert torch.equal(torch.nan_to_num(g, nan=123.0), torch.nan_to_num(w, nan=123.0)), (g.shape, given.keys())
        assert bool(torch.isfinite(got[2]).all()) and got[2].abs().max().item() <= 0.75


@pytest.mark.parametrize("dims,dtype", [((128, 128), "bf16"), ((128, 128, 128, 128), "bf16"), ((128, 512, 512, 128), "bf16"), ((128, 128, 128), "f32"),
                                        ((128, 512, 128), "f32")])
@pytest.mark.parametrize("M", [40, 300, 5000, 40000])
def test_pairs_that_touch_one_anothers_memory_run_one_after_the_other(dims, dtype, M):
    """The second network on the first one's output, the first on rows that the second overwrites, outputs that overlap, and actions that take the place
    of an input: what the calls give one by one, in every form of the pair's launch."""
    from ksim_amd.env_terms import action_sample, sample_action
    from ksim_amd.mlp import MLP

    rng = np.random.default_rng(M)
    a, b = (MLP([rng.normal(scale=i ** -0.5, size=(o, i)) for i, o in zip(dims[:-1], dims[1:])], [0.1 * rng.normal(size=o) for o in dims[1:]],
                activation="elu", dtype=dtype) for _ in range(2))
    n = M * 128
    given = torch.from_numpy(rng.normal(size=4 * n + 64).astype(np.float32)).cuda()
    rows = lambda buf, first: buf[first : first + n].view(M, 128)  # noqa: E731
    for xa, ya, xb, yb in ((0, n, n, 2 * n), (0, n, n + 64, 3 * n), (0, n, 2 * n, 0), (0, n, 3 * n, n + 64), (0, n, 3 * n, n - 64)):
        want, got = given.clone(), given.clone()
        a(rows(want, xa), out=rows(want, ya))
        b(rows(want, xb), out=rows(want, yb))
        a.forward_pair(rows(got, xa), rows(got, ya), b, rows(got, xb), rows(got, yb))
        assert torch.equal(got, want), (xa, ya, xb, yb)
    log_std = torch.full((128,), -1.0, device="cuda")
    for out, noise in ((0, None), (n, None), (2 * n, None), (3 * n, None), (None, n), (None, 3 * n)):
        results = []
        for in_launch in (False, True):
            buf, apart = given.clone(), torch.empty(M, 128, device="cuda")
            sampling = dict(seed=3, clip_max=1.5, out=apart if out is None else rows(buf, out), noise=None if noise is None else rows(buf, noise))
            args = (rows(buf, 0), rows(buf, n), b, rows(buf, 2 * n), rows(buf, 3 * n))
            a.forward_pair(*args, action_sample(args[1], log_std, **sampling) if in_launch else None)
            if not in_launch:
                sample_action(args[1], log_std, **sampling)
            results.append(buf if out is not None else torch.cat([buf, apart.view(-1)]))
        assert torch.equal(*results), (out, noise)


@pytest.mark.parametrize("M", [37, 1544])
def test_layers_that_need_one_another_go_backward_in_their_order(M):
    """A chain of layers whose gradients are one another's operands, a gradient over another's input rows, and one network twice, in one call: what
    the calls give one by one."""
    from ksim_amd.mlp import MLP
    from ksim_amd.recurrent import LayerBackward, run_layers_backward

    rng = np.random.default_rng(M)
    t = lambda *s: torch.from_numpy(rng.normal(size=s).astype(np.float32)).cuda()  # noqa: E731
    nets = []
    for dtype in ("bf16", "bf16", "f32"):
        nets.append(MLP([rng.normal(scale=0.1, size=(128, 128))], [0.1 * rng.normal(size=128)], activation="none", dtype=dtype))
        nets[-1].train_init()
    a, b, c = nets
    x, dy, wide = t(M, 128), t(M, 128), t(M, 160)

    def entries(d1, d2, rows):
        return [[LayerBackward(a, dy, x, d1), LayerBackward(b, d1, x, d2), LayerBackward(c, d2, x)],  # down a chain
                [LayerBackward(a, dy, rows[:, 32:]), LayerBackward(b, dy, None, rows.view(-1)[64:][: M * 128].view(M, 128))],  # over rows read before
                [LayerBackward(b, dy, None, d1), LayerBackward(a, dy, None, d1)],  # one place twice
                [LayerBackward(a, dy, x), LayerBackward(a, x, dy), LayerBackward(c, dy, x)]]  # one gradient twice

    for k in range(4):
        results = []
        for together in (False, True):
            d1, d2, rows = torch.zeros(M, 128, device="cuda"), torch.zeros(M, 128, device="cuda"), wide.clone()
            calls = entries(d1, d2, rows)[k]
            if together:
                run_layers_backward(calls)
            else:
                for call in calls:
                    run_layers_backward([call])
            results.append([d1, d2, rows] + [g for net in nets for pair in net.parameters(gradients=True) for g in pair])
        assert all(torch.equal(u, v) for u, v in zip(*results)), k


@pytest.mark.parametrize("M", [37, 1544])
def test_layers_too_wide_for_the_whole_network_kernel_in_shared_launches(M):
    """A bf16 layer of more outputs than the whole-network kernel holds takes its input gradient through the call's workspace, which the weight
    gradients of all layers use behind it; more weight gradients of one precision than a launch's table takes beside them."""
    from ksim_amd.mlp import MLP
    from ksim_amd.recurrent import LayerBackward, run_layers_backward

    rng = np.random.default_rng(M)
    t = lambda *s: torch.from_numpy(rng.normal(size=s).astype(np.float32)).cuda()  # noqa: E731
    results, shapes = [], [(128, 768), (128, 384), (256, 768), (128, 2048)] + [(43, 128)] * 10
    nets = [MLP([rng.normal(scale=i ** -0.5, size=(o, i))], [0.1 * rng.normal(size=o)], activation="none", dtype="bf16") for i, o in shapes]
    rows = [(t(M, n.in_dim), t(M, n.out_dim)) for n in nets]
    for n in nets:
        n.train_init()
    for together in (False, True):
        dxs = [torch.empty(M, n.in_dim, device="cuda") for n in nets]
        for n, (x, dy), dx in zip(nets, rows, dxs):
            if together:
                n.layer_weight_grad(dy.new_ones(M, n.in_dim), torch.ones_like(dy))  # something else in the handle
            else:
                n.backward_dx(x, dy, dx)
        if together:
            run_layers_backward([LayerBackward(n, dy, x, dx) for n, (x, dy), dx in zip(nets, rows, dxs)])
        results.append(dxs + [g.clone() for n in nets for pair in n.parameters(gradients=True) for g in pair])
    assert all(torch.equal(a, b) for a, b in zip(*results))
