"""GRU cell and recurrent policy networks on the GPU against the float64 oracle."""
import numpy as np
import pytest
import torch

from oracle import recurrent as orec

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def t32(a):
    return torch.tensor(np.asarray(a), dtype=torch.float32, device=DEV).contiguous()


def _bf16(a):
    return torch.tensor(np.asarray(a), dtype=torch.float32).bfloat16().double().numpy()


def _cell_params(rng, I, H):
    s = 1.0 / np.sqrt(H)
    return (rng.uniform(-s, s, (3 * H, I)), rng.uniform(-s, s, (3 * H, H)), rng.uniform(-s, s, 3 * H), rng.uniform(-s, s, H))


@pytest.mark.parametrize("N,I,H", [(33, 20, 24), (512, 128, 128), (8192, 256, 256)])
def test_gru_cell_f32_and_bf16(N, I, H):
    from ksim_amd.recurrent import GRUCell

    rng = np.random.default_rng(N)
    wi, wh, b, bn = _cell_params(rng, I, H)
    x, h = rng.normal(size=(N, I)), rng.normal(size=(N, H)) * 0.5
    fresh = rng.random(N) < 0.2
    h_eff = np.where(fresh[:, None], 0.0, h)
    want = orec.gru_cell(x, h_eff, wi, wh, b, bn)
    mask = torch.from_numpy(fresh.astype(np.uint8)).to(DEV)
    got = GRUCell(wi, wh, b, bn, dtype="f32")(t32(x), t32(h), mask).cpu().numpy()
    np.testing.assert_allclose(got, want, rtol=2e-5, atol=2e-5)  # fp32 projections vs float64
    # bf16 projections: operands of the two matrix products rounded to bf16, everything else fp32
    gi = _bf16(x) @ _bf16(wi).T + b
    gh = _bf16(h) @ _bf16(wh).T
    gh = np.where(fresh[:, None], 0.0, gh)
    r = orec.sigmoid(gi[:, :H] + gh[:, :H]); z = orec.sigmoid(gi[:, H:2 * H] + gh[:, H:2 * H])
    n = np.tanh(gi[:, 2 * H:] + r * (gh[:, 2 * H:] + bn))
    want16 = n + z * (h_eff - n)
    cell = GRUCell(wi, wh, b, bn, dtype="bf16")
    hin = t32(h)
    got16 = cell(t32(x), hin, mask, out=hin).cpu().numpy()  # in place on the carry
    np.testing.assert_allclose(got16, want16, rtol=2e-4, atol=2e-4)
    assert np.abs(got16 - want).max() < 3e-2  # and close to the unrounded cell
    # no bias, no mask
    got0 = GRUCell(wi, wh, dtype="f32")(t32(x), t32(h)).cpu().numpy()
    np.testing.assert_allclose(got0, orec.gru_cell(x, h, wi, wh), rtol=2e-5, atol=2e-5)


def test_recurrent_network_over_an_episode_with_restarts():
    """Input projection, two GRU layers and a GELU output MLP stepped ten times; some envs restart along the way."""
    from ksim_amd.mlp import MLP
    from ksim_amd.recurrent import GRUCell, RecurrentNetwork

    rng = np.random.default_rng(5)
    N, I, H, O, depth = 96, 43, 64, 60, 2
    proj = (rng.normal(size=(H, I)) / np.sqrt(I), rng.normal(size=H) * 0.1)
    cells = [_cell_params(rng, H, H) for _ in range(depth)]
    ow = [rng.normal(size=(H, H)) / np.sqrt(H), rng.normal(size=(O, H)) / np.sqrt(H)]
    ob_ = [rng.normal(size=H) * 0.1, np.zeros(O)]  # use_final_bias=False (walking.py:98-106)
    net = RecurrentNetwork(proj, [GRUCell(*c, dtype="f32") for c in cells], MLP(ow, ob_, activation="gelu", dtype="f32"), dtype="f32")
    carry = net.initial_carry(N, DEV)
    want_carry = np.zeros((depth, N, H))
    for k in range(10):
        obs = rng.normal(size=(N, I))
        fresh = rng.random(N) < (0.0 if k == 0 else 0.15)
        out = net(t32(obs), carry, torch.from_numpy(fresh.astype(np.uint8)).to(DEV))
        want, want_carry = orec.recurrent_network(obs, want_carry, fresh, proj, cells, ow, ob_)
        np.testing.assert_allclose(out.cpu().numpy(), want, rtol=1e-4, atol=1e-4)
        np.testing.assert_allclose(carry.cpu().numpy(), want_carry, rtol=1e-4, atol=1e-4)
    with pytest.raises(Exception, match="carry"):
        net(t32(obs), carry[:1])


def test_gelu_mlp_bf16():
    from ksim_amd.mlp import MLP

    rng = np.random.default_rng(6)
    dims = (64, 256, 256, 40)
    ws = [rng.normal(size=(o, i)) / np.sqrt(i) for i, o in zip(dims[:-1], dims[1:])]
    bs = [rng.normal(size=o) * 0.1 for o in dims[1:]]
    for M in (100, 40000):  # the per-layer and the whole-network kernels
        x = rng.normal(size=(M, dims[0]))
        got = MLP(ws, bs, activation="gelu", dtype="bf16")(t32(x)).cpu().numpy()
        h = _bf16(x)
        for i, (w, b) in enumerate(zip(ws, bs)):
            h = h @ _bf16(w).T + b
            if i + 1 < len(ws):
                h = _bf16(orec.gelu(h))
        assert np.abs(got - h).max() < 6e-3 * max(1.0, np.abs(h).max())
        got32 = MLP(ws, bs, activation="gelu", dtype="f32")(t32(x)).cpu().numpy()
        np.testing.assert_allclose(got32, orec.mlp(x, ws, bs, orec.gelu), rtol=2e-5, atol=2e-5)


@pytest.mark.parametrize("N,I,H", [(40, 12, 16), (4096, 128, 128)])
def test_lstm_cell_and_network(N, I, H):
    from ksim_amd.mlp import MLP
    from ksim_amd.recurrent import LSTMCell, RecurrentNetwork

    rng = np.random.default_rng(N + 1)
    s = 1.0 / np.sqrt(H)
    def params(i):
        return (rng.uniform(-s, s, (4 * H, i)), rng.uniform(-s, s, (4 * H, H)), rng.uniform(-s, s, 4 * H))
    wi, wh, b = params(I)
    x, h, c = rng.normal(size=(N, I)), rng.normal(size=(N, H)) * 0.5, rng.normal(size=(N, H))
    fresh = rng.random(N) < 0.25
    keep = ~fresh[:, None]
    hw, cw = orec.lstm_cell(x, h * keep, c * keep, wi, wh, b)
    mask = torch.from_numpy(fresh.astype(np.uint8)).to(DEV)
    hg, cg = LSTMCell(wi, wh, b, dtype="f32")(t32(x), t32(h), t32(c), mask)
    np.testing.assert_allclose(hg.cpu().numpy(), hw, rtol=2e-5, atol=2e-5)
    np.testing.assert_allclose(cg.cpu().numpy(), cw, rtol=2e-5, atol=2e-5)
    hg, cg = LSTMCell(wi, wh, b, dtype="bf16")(t32(x), t32(h), t32(c), mask)
    assert np.abs(hg.cpu().numpy() - hw).max() < 3e-2 and np.abs(cg.cpu().numpy() - cw).max() < 5e-2
    # the K-Bot actor's shape: projection, two LSTM layers, ELU output MLP; carry (depth, 2, N, H) advanced in place
    proj = (rng.normal(size=(H, I)) / np.sqrt(I), rng.normal(size=H) * 0.1)
    cells = [params(H) for _ in range(2)]
    ow, ob_ = [rng.normal(size=(H, H)) / np.sqrt(H), rng.normal(size=(40, H)) / np.sqrt(H)], [rng.normal(size=H) * 0.1, np.zeros(40)]
    net = RecurrentNetwork(proj, [LSTMCell(*p, dtype="f32") for p in cells], MLP(ow, ob_, activation="elu", dtype="f32"), dtype="f32")
    carry = net.initial_carry(N, DEV)
    assert tuple(carry.shape) == (2, 2, N, H)
    want_carry = np.zeros((2, 2, N, H))
    elu = lambda v: np.where(v > 0, v, np.expm1(v))  # noqa: E731
    for k in range(6):
        obs = rng.normal(size=(N, I))
        fr = rng.random(N) < (0.0 if k == 0 else 0.2)
        out = net(t32(obs), carry, torch.from_numpy(fr.astype(np.uint8)).to(DEV))
        want, want_carry = orec.recurrent_network(obs, want_carry, fr, proj, cells, ow, ob_, act=elu)
        np.testing.assert_allclose(out.cpu().numpy(), want, rtol=2e-4, atol=2e-4)
        np.testing.assert_allclose(carry.cpu().numpy(), want_carry, rtol=2e-4, atol=2e-4)


@pytest.mark.parametrize("dtype,tol,act", [("f32", 2e-4, "elu"), ("bf16", 6e-2, "elu"), ("f32", 2e-4, "gelu")])
def test_backward_through_time_matches_the_oracle(dtype, tol, act):
    _check_backward_through_time(dtype, tol, act, 64, 96)


@pytest.mark.parametrize("dtype,tol", [("f32", 2e-4), ("bf16", 6e-2)])
@pytest.mark.parametrize("N", [77, 16])
def test_backward_through_time_of_the_sequence_kernels_matches_the_oracle(dtype, tol, N):
    """Hidden size 128: one launch per trajectory and direction (`ks_gru_sequence_*`), rows that do not fill the last set of four."""
    _check_backward_through_time(dtype, tol, "elu", 128, N)


def _check_backward_through_time(dtype, tol, act, H, N):
    """Gradients of a GRU actor over a trajectory (input projection, two GRU layers, ELU or GELU output network) with episode
    starts inside it, against torch float64 reverse-mode differentiation of the oracle network; then one optimiser step.
    Tolerances are relative to the largest entry of each gradient array: fp32 accumulation only for f32; for bf16 the
    activations and the gradients between layers are rounded to bf16 at every one of the T steps."""
    from ksim_amd import _lib_terms as T
    from ksim_amd.mlp import MLP
    from ksim_amd.recurrent import GRUCell, RecurrentNetwork

    rng = np.random.default_rng(41)
    Tn, I, O = 12, 37, 10
    proj = (rng.normal(size=(H, I)) / np.sqrt(I), rng.normal(size=H) * 0.1)
    cells = [(rng.normal(size=(3 * H, H)) / np.sqrt(H), rng.normal(size=(3 * H, H)) / np.sqrt(H), rng.normal(size=3 * H) * 0.1,
              rng.normal(size=H) * 0.1) for _ in range(2)]
    ow = [rng.normal(size=(H, H)) / np.sqrt(H), rng.normal(size=(O, H)) / np.sqrt(H)]
    ob = [rng.normal(size=H) * 0.1, rng.normal(size=O) * 0.1]
    obs, carry0 = rng.normal(size=(Tn, N, I)), rng.normal(size=(2, N, H)) * 0.5
    fresh = rng.random((Tn, N)) < 0.08
    d_out = rng.normal(size=(Tn, N, O))
    if dtype == "bf16":  # both sides start from bf16-representable weights
        rb = lambda a: torch.tensor(a, dtype=torch.float32).to(torch.bfloat16).to(torch.float64).numpy()  # noqa: E731
        proj = (rb(proj[0]), proj[1]); ow = [rb(w) for w in ow]
        cells = [(rb(c[0]), rb(c[1]), c[2], c[3]) for c in cells]
    want_out, want = orec.recurrent_sequence_gradients(obs, carry0, fresh, proj, cells, ow, ob, d_out, act=act)

    net = RecurrentNetwork(proj, [GRUCell(*c, dtype=dtype) for c in cells], MLP(ow, ob, activation=act, dtype=dtype), dtype=dtype)
    net.train_init()
    assert all(c.sequence_supported == (H == 128) for c in net.cells)
    out = net.train_forward(t32(obs), t32(carry0), torch.tensor(fresh, dtype=torch.uint8, device=DEV))
    scale = np.abs(want_out).max()
    assert np.abs(out.cpu().numpy() - want_out).max() <= (1e-4 if dtype == "f32" else 3e-2) * scale
    net.backward(t32(d_out))
    got = {"input_proj.W": net.input_proj.parameters(True)[0][0], "input_proj.b": net.input_proj.parameters(True)[0][1]}
    ref = {"input_proj.W": want["input_proj"][0], "input_proj.b": want["input_proj"][1]}
    for i, c in enumerate(net.cells):
        g = c.parameters(True)
        for k, j in (("weight_ih", 0), ("weight_hh", 1), ("bias", 2), ("bias_n", 3)):
            got[f"cell{i}.{k}"], ref[f"cell{i}.{k}"] = g[k], want["cells"][i][j]
    for l, (w, b) in enumerate(net.output_proj.parameters(True)):
        got[f"out{l}.W"], ref[f"out{l}.W"], got[f"out{l}.b"], ref[f"out{l}.b"] = w, want["out"][l][0], b, want["out"][l][1]
    for k in ref:
        err = np.abs(got[k].cpu().numpy() - ref[k]).max() / np.abs(ref[k]).max()
        assert err <= tol, f"{k}: {err:.2e} > {tol}"
    # the hidden projection has no reset / update bias of its own: those entries stay out of the update
    before = [c.parameters() for c in net.cells]
    acc = torch.zeros(1, dtype=torch.float64, device=DEV)
    net.grad_sqnorm(acc)
    total = sum(float((np.asarray(v) ** 2).sum()) for v in ref.values())
    assert acc.item() == pytest.approx(total, rel=2e-3 if dtype == "f32" else 0.15)
    params = T.KsAdamParams(1e-3, 0.9, 0.999, 1e-8, 0.0, 0.0, 1)
    net.adam_step(params, None)
    for c, b0 in zip(net.cells, before):
        p = c.parameters()
        (_, bh), = c.proj_h.parameters()
        assert torch.equal(bh[:2 * H], torch.zeros(2 * H, device=DEV))
        # first Adam step: every parameter with a gradient moves by lr against the gradient's sign
        moved = (p["bias_n"] - b0["bias_n"]).cpu().numpy()
        gn = c.parameters(True)["bias_n"].cpu().numpy()
        big = np.abs(gn) > 1e-4
        np.testing.assert_allclose(moved[big], -1e-3 * np.sign(gn[big]), rtol=1e-3)
    # the forward pass of the rollout sees the updated b_n also for envs that start an episode
    h1 = net.cells[0](t32(rng.normal(size=(N, H))), t32(np.zeros((N, H))), torch.ones(N, dtype=torch.uint8, device=DEV))
    assert torch.isfinite(h1).all()


@pytest.mark.parametrize("dtype,tol,H,N", [("f32", 2e-4, 64, 80), ("bf16", 6e-2, 64, 80), ("f32", 2e-4, 128, 77), ("f32", 2e-4, 128, 16)])
def test_lstm_backward_through_time_matches_the_oracle(dtype, tol, H, N):
    """The same for an LSTM stack (the K-Bot example's actor shape: projection, LSTM layers, linear output).  Hidden size
    128 in fp32 is the K-Bot cell itself and runs through the one-launch-per-trajectory kernels (`ks_lstm_sequence_*`),
    with a row count that does not fill the last 16-row workgroup."""
    from ksim_amd import _lib_terms as T
    from ksim_amd.mlp import MLP
    from ksim_amd.recurrent import LSTMCell, RecurrentNetwork

    rng = np.random.default_rng(43)
    Tn, I, O = 10, 29, 12
    proj = (rng.normal(size=(H, I)) / np.sqrt(I), rng.normal(size=H) * 0.1)
    cells = [(rng.normal(size=(4 * H, H)) / np.sqrt(H), rng.normal(size=(4 * H, H)) / np.sqrt(H), rng.normal(size=4 * H) * 0.1)
             for _ in range(2)]
    ow, ob = [rng.normal(size=(O, H)) / np.sqrt(H)], [rng.normal(size=O) * 0.1]
    obs, carry0 = rng.normal(size=(Tn, N, I)), rng.normal(size=(2, 2, N, H)) * 0.5
    fresh = rng.random((Tn, N)) < 0.08
    d_out = rng.normal(size=(Tn, N, O))
    if dtype == "bf16":
        proj = (_bf16(proj[0]), proj[1]); ow = [_bf16(w) for w in ow]
        cells = [(_bf16(c[0]), _bf16(c[1]), c[2]) for c in cells]
    want_out, want = orec.recurrent_sequence_gradients(obs, carry0, fresh, proj, cells, ow, ob, d_out)
    net = RecurrentNetwork(proj, [LSTMCell(*c, dtype=dtype) for c in cells], MLP(ow, ob, activation="none", dtype=dtype), dtype=dtype)
    net.train_init()
    assert all(c.sequence_supported == (dtype == "f32" and H == 128) for c in net.cells)
    out = net.train_forward(t32(obs), t32(carry0), torch.tensor(fresh, dtype=torch.uint8, device=DEV))
    assert np.abs(out.cpu().numpy() - want_out).max() <= (1e-4 if dtype == "f32" else 3e-2) * np.abs(want_out).max()
    net.backward(t32(d_out))
    got = {"input_proj.W": net.input_proj.parameters(True)[0][0], "input_proj.b": net.input_proj.parameters(True)[0][1],
           "out.W": net.output_proj.parameters(True)[0][0], "out.b": net.output_proj.parameters(True)[0][1]}
    ref = {"input_proj.W": want["input_proj"][0], "input_proj.b": want["input_proj"][1], "out.W": want["out"][0][0], "out.b": want["out"][0][1]}
    for i, c in enumerate(net.cells):
        g = c.parameters(True)
        for k, j in (("weight_ih", 0), ("weight_hh", 1), ("bias", 2)):
            got[f"cell{i}.{k}"], ref[f"cell{i}.{k}"] = g[k], want["cells"][i][j]
    for k in ref:
        err = np.abs(got[k].cpu().numpy() - ref[k]).max() / np.abs(ref[k]).max()
        assert err <= tol, f"{k}: {err:.2e} > {tol}"
    net.adam_step(T.KsAdamParams(1e-3, 0.9, 0.999, 1e-8, 0.0, 0.0, 1), None)
    for c in net.cells:  # the hidden projection carries no bias of its own, before and after the update
        (_, bh), = c.proj_h.parameters()
        assert torch.equal(bh, torch.zeros(4 * H, device=DEV))


def test_lstm_sequence_kernels_agree_with_the_step_by_step_entry_points():
    """One launch over the trajectory against T calls of the per-step entry points on the same cell (which, for such a cell,
    are that launch with T = 1): states, saved activations and gate gradients bit for bit; the carry of the hidden-state
    gradient, which the per-step path forms with a separate product, to rounding.  In place with T = 1, as the rollout
    advances its carry."""
    from ksim_amd import _lib
    from ksim_amd.recurrent import LSTMCell

    rng = np.random.default_rng(47)
    Tn, M, H = 7, 45, 128
    cell = LSTMCell(rng.normal(size=(4 * H, H)) / np.sqrt(H), rng.normal(size=(4 * H, H)) / np.sqrt(H), rng.normal(size=4 * H) * 0.1, dtype="f32")
    cell.train_init()
    assert cell.sequence_supported
    x, h0, c0 = t32(rng.normal(size=(Tn, M, H))), t32(rng.normal(size=(M, H)) * 0.5), t32(rng.normal(size=(M, H)) * 0.5)
    fresh = torch.tensor(rng.random((Tn, M)) < 0.1, dtype=torch.uint8, device=DEV)
    z = lambda *s: torch.zeros(*s, device=DEV)  # noqa: E731
    hs, cs, sv = z(Tn, M, H), z(Tn, M, H), z(Tn, M, 7 * H)
    cell.sequence_forward(x, h0, c0, fresh, hs, cs, sv)
    hs1, cs1, sv1 = z(Tn, M, H), z(Tn, M, H), z(Tn, M, 7 * H)
    for t in range(Tn):
        cell.train_forward(x[t], h0 if t == 0 else hs1[t - 1], c0 if t == 0 else cs1[t - 1], fresh[t], hs1[t], cs1[t], sv1[t])
    assert torch.equal(hs, hs1) and torch.equal(cs, cs1) and torch.equal(sv, sv1)
    h, c = h0.clone(), c0.clone()  # the rollout's step: the carry advanced in place
    for t in range(Tn):
        cell(x[t], h, c, fresh[t], out=(h, c))
    assert torch.equal(h, hs[-1]) and torch.equal(c, cs[-1])
    dH = t32(rng.normal(size=(Tn, M, H)))
    d_g = z(Tn, M, 4 * H)
    cell.sequence_backward(dH, sv, fresh, d_g)
    d_g1, carry, ccarry = z(Tn, M, 4 * H), z(2, M, H), z(2, M, H)
    dH1 = dH.clone()
    for t in range(Tn - 1, -1, -1):
        dH1[t] += carry[t & 1]
        cell.backward_step(dH1[t], ccarry[t & 1], sv[t], fresh[t], d_g1[t], carry[(t + 1) & 1], ccarry[(t + 1) & 1])
    err = (d_g - d_g1).abs().max().item() / d_g1.abs().max().item()
    assert err < 1e-5, err
    assert torch.equal(d_g[-1], d_g1[-1])  # the last step has no carried gradient yet: the same arithmetic
    lib = _lib.load()  # shapes the kernels do not cover are refused, not approximated
    small = LSTMCell(rng.normal(size=(4 * 64, 64)), rng.normal(size=(4 * 64, 64)), None, dtype="f32")
    assert not small.sequence_supported
    assert lib.ks_lstm_sequence_forward(small._handle, _lib.current_stream(), 1, 4, _lib.ptr(z(4, 256)), _lib.ptr(z(4, 64)), _lib.ptr(z(4, 64)),
                                        None, _lib.ptr(z(4, 64)), None, None) != 0
    assert lib.ks_lstm_sequence_forward(cell._handle, _lib.current_stream(), 2, M, _lib.ptr(z(2, M, 4 * H)), _lib.ptr(h0), _lib.ptr(c0),
                                        None, _lib.ptr(h0), None, None) != 0  # aliasing is for T = 1 only


def test_lstm_sequence_forward_over_many_rows_equals_the_same_rows_in_small_calls():
    """A short call over thousands of rows lets each workgroup take several 4-row sets in turn (the rollout's single step over all
    envs): the rows must come out exactly as when they are given in calls small enough for one set per workgroup, including a
    last set that is not full, in place as the rollout calls it, and with the episode starts honoured."""
    from ksim_amd.recurrent import LSTMCell

    rng = np.random.default_rng(53)
    M, H = 2102, 128
    cell = LSTMCell(rng.normal(size=(4 * H, H)) / np.sqrt(H), rng.normal(size=(4 * H, H)) / np.sqrt(H), rng.normal(size=4 * H) * 0.1, dtype="f32")
    cell.train_init()
    z = lambda *s: torch.zeros(*s, device=DEV)  # noqa: E731
    for Tn in (1, 3):
        x, h0, c0 = t32(rng.normal(size=(Tn, M, H))), t32(rng.normal(size=(M, H)) * 0.5), t32(rng.normal(size=(M, H)) * 0.5)
        fresh = torch.tensor(rng.random((Tn, M)) < 0.1, dtype=torch.uint8, device=DEV)
        hs, cs, sv = z(Tn, M, H), z(Tn, M, H), z(Tn, M, 7 * H)
        cell.sequence_forward(x, h0, c0, fresh, hs, cs, sv)
        for lo in range(0, M, 700):
            hi = min(M, lo + 700)
            n = hi - lo
            hs1, cs1, sv1 = z(Tn, n, H), z(Tn, n, H), z(Tn, n, 7 * H)
            cell.sequence_forward(x[:, lo:hi].contiguous(), h0[lo:hi].contiguous(), c0[lo:hi].contiguous(), fresh[:, lo:hi].contiguous(),
                                  hs1, cs1, sv1)
            assert torch.equal(hs[:, lo:hi], hs1) and torch.equal(cs[:, lo:hi], cs1) and torch.equal(sv[:, lo:hi], sv1), (Tn, lo)
    h, c = h0.clone(), c0.clone()  # one step in place over all rows, as the rollout advances its carry
    cell(x[0], h, c, fresh[0], out=(h, c))
    hs1, cs1, sv1 = z(1, M, H), z(1, M, H), z(1, M, 7 * H)
    cell.sequence_forward(x[:1].contiguous(), h0, c0, fresh[:1].contiguous(), hs1, cs1, sv1)
    assert torch.equal(h, hs1[0]) and torch.equal(c, cs1[0])


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("Tn,M", [(1, 1), (7, 45), (3, 2102)])
def test_gru_sequence_kernels_agree_with_the_step_by_step_entry_points(dtype, Tn, M):
    """One launch over the trajectory against T calls of the per-step entry points: states and saved activations bit for bit
    (for such a cell a step is that launch with T = 1), gate gradients against the per-step backward, whose product is a kernel of
    its own: to fp32 rounding, and for bf16 cells to its rounding of every step's product to bf16 (2^-9 of the largest per step).
    Rows that do not fill the last 4-row set, and enough of them for several sets per workgroup."""
    from ksim_amd.recurrent import GRUCell

    rng = np.random.default_rng(59)
    H = 128
    cell = GRUCell(*_cell_params(rng, H, H), dtype=dtype)
    assert cell.sequence_supported
    cell.train_init()
    x, h0 = t32(rng.normal(size=(Tn, M, H))), t32(rng.normal(size=(M, H)) * 0.5)
    fresh = torch.tensor(rng.random((Tn, M)) < 0.1, dtype=torch.uint8, device=DEV)
    z = lambda *s: torch.zeros(*s, device=DEV)  # noqa: E731
    hs, sv = z(Tn, M, H), z(Tn, M, 5 * H)
    cell.sequence_forward(x, h0, fresh, hs, sv)
    hs1, sv1, h = z(Tn, M, H), z(Tn, M, 5 * H), h0.clone()
    for t in range(Tn):
        cell.train_forward(x[t], h0 if t == 0 else hs1[t - 1], fresh[t], hs1[t], sv1[t])
        cell(x[t], h, fresh[t], out=h)  # the rollout's step: the carry advanced in place
    assert torch.equal(hs, hs1) and torch.equal(sv, sv1) and torch.equal(h, hs[-1])
    dH = t32(rng.normal(size=(Tn, M, H)))
    d_gi, d_gh, d_gi1, d_gh1, carry, dH1 = z(Tn, M, 3 * H), z(Tn, M, 3 * H), z(Tn, M, 3 * H), z(Tn, M, 3 * H), z(2, M, H), dH.clone()
    cell.sequence_backward(dH, sv, fresh, d_gi, d_gh)
    for t in range(Tn - 1, -1, -1):
        dH1[t] += carry[t & 1]
        cell.backward_step(dH1[t], sv[t], fresh[t], d_gi1[t], d_gh1[t], carry[(t + 1) & 1])
    tol = 1e-5 if dtype == "f32" else Tn * 2.0 ** -9
    for got, want in ((d_gi, d_gi1), (d_gh, d_gh1)):
        assert (got - want).abs().max().item() <= tol * want.abs().max().item()
    assert not GRUCell(*_cell_params(rng, 24, 24), dtype=dtype).sequence_supported


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("H", [128, 24])
def test_gru_gates_are_accurate_to_the_last_bits(dtype, H):
    """The gates against float64, one input each: a candidate of size 1e-6 has the relative error of one of size 1, and so have the sigmoids far
    out.  Library functions and IEEE division stay within 4 ulp (2^-22); 1 - 2 / (e^2x + 1) would lose three digits at 1e-4."""
    from ksim_amd.recurrent import GRUCell

    v = np.concatenate([np.logspace(-6, 1.3, 200), np.linspace(0.01, 85.0, 184)])
    v = np.concatenate([v, -v])
    if dtype == "bf16":
        v = _bf16(v)
    x = np.resize(v, (v.size, H)).astype(np.float32)
    for shift in range(x.shape[0]):  # every unit of the cell meets every value
        x[shift] = np.resize(np.roll(v, shift), H)
    eye = np.eye(H)
    zero = np.zeros((H, H))
    M = x.shape[0]
    fresh = torch.ones(M, dtype=torch.uint8, device=DEV)
    xt, h0 = t32(x), torch.zeros(M, H, device=DEV)
    for gate in range(3):
        wi = np.concatenate([eye if g == gate else zero for g in range(3)])
        cell = GRUCell(wi, np.zeros((3 * H, H)), dtype=dtype)
        cell.train_init()
        out, saved = torch.empty(M, H, device=DEV), torch.empty(M, 5 * H, device=DEV)
        cell.train_forward(xt, h0, fresh, out, saved)
        got = saved[:, gate * H:(gate + 1) * H].double().cpu().numpy()
        x64 = x.astype(np.float64)
        want = np.tanh(x64) if gate == 2 else 1 / (1 + np.exp(-x64))
        err = np.abs(got - want) / np.abs(want)
        assert err.max() <= 2.0 ** -22, (gate, err.max(), x.ravel()[err.argmax()])


@pytest.mark.parametrize("kind", ["gru", "lstm"])
def test_sequence_without_a_backward_pass_is_bounded_in_memory(kind, monkeypatch):
    """A trajectory longer than what is kept at a time goes through in stretches of steps, from carry to carry: the same bits as in one piece and as
    step by step, and scratch that does not grow with the number of steps."""
    from ksim_amd import recurrent
    from ksim_amd.mlp import random_mlp

    rng = np.random.default_rng(61)
    Tn, M, H, I = 37, 45, 128, 19
    G, cls = (3, recurrent.GRUCell) if kind == "gru" else (4, recurrent.LSTMCell)
    cells = [cls(rng.normal(size=(G * H, H)) / np.sqrt(H), rng.normal(size=(G * H, H)) / np.sqrt(H), rng.normal(size=G * H) * 0.1, dtype="f32")
             for _ in range(2)]
    out, _, _ = random_mlp((H, 7), 3, activation="none", dtype="f32")
    net = recurrent.RecurrentNetwork((rng.normal(size=(H, I)) / np.sqrt(I), np.zeros(H)), cells, out, dtype="f32")
    obs = t32(rng.normal(size=(Tn, M, I)))
    carry = t32(rng.normal(size=net.initial_carry(M).shape) * 0.5)
    kept = carry.clone()
    fresh = torch.tensor(rng.random((Tn, M)) < 0.1, dtype=torch.uint8, device=DEV)
    want, c = torch.empty(Tn, M, 7, device=DEV), carry.clone()
    for t in range(Tn):
        net(obs[t], c, fresh=fresh[t], out=want[t])
    strided = torch.stack([obs, obs], 2)[:, :, 0]  # not contiguous
    for rows in (10 ** 9, 5 * M, 5 * M - 1, M, 1):  # the last: less than a step, which is then a stretch of its own
        monkeypatch.setattr(recurrent, "SEQUENCE_ROWS", rows)
        for o in (obs, strided):
            assert torch.equal(net.forward_sequence(o, carry, fresh), want)
        assert torch.equal(carry, kept)
    monkeypatch.undo()
    Tn, M = 64, 16384
    obs = torch.randn(Tn, M, I, device=DEV)
    carry, fresh = net.initial_carry(M), torch.zeros(Tn, M, dtype=torch.uint8, device=DEV)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    net.forward_sequence(obs, carry, fresh)
    # the output, and for each row of a stretch the input, projected input, hidden and cell state of a layer and the next layer's
    assert torch.cuda.max_memory_allocated() - before <= Tn * M * 7 * 4 + recurrent.SEQUENCE_ROWS * (4 + G) * H * 4 + (1 << 24)


@pytest.mark.parametrize("kind,dtype", [("lstm", "f32"), ("gru", "f32"), ("gru", "bf16")])
@pytest.mark.parametrize("rows,steps", [((1, 6), 3), ((1030, 37), 5), ((4, 1), 2), ((2500, 8), 1)])
def test_two_layers_in_one_launch_match_one_by_one(kind, dtype, rows, steps):
    """The actor's and the critic's layer of a depth share a launch: other weights, other row counts (ragged sets of 4), several sets
    per workgroup for the short call, against the same layers launched by themselves, forward and backward, bit for bit."""
    from ksim_amd.recurrent import GRUCell, LSTMCell, run_sequences

    H, G, S = 128, 4 if kind == "lstm" else 3, 7 if kind == "lstm" else 5
    rng = np.random.default_rng(sum(rows) + steps)
    cells, forward, backward, want = [], [], [], []
    for M in rows:
        w = [rng.normal(scale=H ** -0.5, size=s) for s in ((G * H, H), (G * H, H), (G * H,))]
        cell = LSTMCell(*w, dtype=dtype) if kind == "lstm" else GRUCell(*w, 0.1 * rng.normal(size=H), dtype=dtype)
        cell.train_init()
        t = lambda *s: torch.from_numpy(rng.normal(size=s).astype(np.float32)).cuda()  # noqa: E731
        x, h0, c0, dH = t(steps, M, H), t(M, H), t(M, H), t(steps, M, H)
        fresh = torch.from_numpy((rng.random((steps, M)) < 0.2).astype(np.uint8)).cuda()
        z = lambda n: torch.full((steps, M, n), 3.0, device="cuda")  # noqa: E731
        state = lambda: (z(H), z(H), z(S * H)) if kind == "lstm" else (z(H), z(S * H))  # noqa: E731
        grads = lambda: (z(G * H),) if kind == "lstm" else (z(G * H), z(G * H))  # noqa: E731
        carry = (h0, c0) if kind == "lstm" else (h0,)
        (*a, sa), (*b, sb), ga, gb = state(), state(), grads(), grads()
        cell.sequence_forward(x, *carry, fresh, *a, sa)
        cell.sequence_backward(dH, sa, fresh, *ga)
        forward.append(cell.sequence_call(x, *carry, fresh, *b, sb))
        backward.append(cell.sequence_backward_call(dH, sb, fresh, *gb))
        want += zip((*a, sa, *ga), (*b, sb, *gb))
        cells.append(cell)
    run_sequences(forward)
    run_sequences(backward)
    for k, (a, b) in enumerate(want):
        assert torch.equal(a, b), k


@pytest.mark.parametrize("rows,steps", [((5, 6), 1), ((1, 37), 2), ((45, 4), 3), ((7, 2), 4)])
def test_lstm_sequences_write_the_outputs_they_are_given_and_no_others(rows, steps):
    """Cell states and saved activations are optional, and each combination is a kernel of its own: states bit for bit those of the call
    that writes everything, for two layers of one call whose outputs differ, with ragged sets of 4 rows and odd and even step counts."""
    from ksim_amd.recurrent import LSTMCell, run_sequences

    H = 128
    rng = np.random.default_rng(71 + steps)
    t = lambda *s: torch.from_numpy(rng.normal(size=s).astype(np.float32)).cuda()  # noqa: E731
    layers = []
    for M in rows:
        cell = LSTMCell(*(rng.normal(scale=H ** -0.5, size=s) for s in ((4 * H, H), (4 * H, H), (4 * H,))), dtype="f32")
        x, h0, c0 = t(steps, M, H), t(M, H), t(M, H)
        fresh = torch.from_numpy((rng.random((steps, M)) < 0.2).astype(np.uint8)).cuda()
        want = [torch.full((steps, M, n * H), 3.0, device="cuda") for n in (1, 1, 7)]
        cell.sequence_forward(x, h0, c0, fresh, *want)
        layers.append((cell, (x, h0, c0, fresh), want))
    kinds = [(cs, sv) for cs in (False, True) for sv in (False, True)]
    for k, first in enumerate(kinds):
        calls, pairs = [], []
        for (cell, given, want), (cs, sv) in zip(layers, (first, kinds[(k + 1) % 4])):
            got = [torch.full_like(w, 5.0) if on else None for w, on in zip(want, (True, cs, sv))]
            calls.append(cell.sequence_call(*given, *got))
            pairs += [(g, w) for g, w in zip(got, want) if g is not None]
        run_sequences(calls)
        for g, w in pairs:
            assert torch.equal(g, w), (k, tuple(w.shape))


@pytest.mark.parametrize("inputs,hidden", [(4, 1), (5, 85), (130, 128), (7, 171), (3, 256), (9, 300)])
def test_parameters_of_a_gru_cell_as_they_were_given(inputs, hidden):
    """The hidden projection's bias leaves from its last third on: inside, at and past the edge of a block."""
    import ctypes

    from ksim_amd import _lib
    from ksim_amd.recurrent import GRUCell

    rng = np.random.default_rng(hidden)
    given = {k: rng.normal(size=n).astype(np.float32) for k, n in
             dict(weight_ih=(3 * hidden, inputs), weight_hh=(3 * hidden, hidden), bias=3 * hidden, bias_n=hidden).items()}
    cell = GRUCell(**given, dtype="f32")
    cell.train_init()
    got = cell.parameters()
    assert got.keys() == given.keys()
    for k, v in given.items():
        assert np.array_equal(got[k].cpu().numpy(), v) and got[k]._base is None
    out = torch.empty(3 * hidden * max(inputs, hidden), device="cuda")
    one = lambda x: (ctypes.c_void_p * 1)(x)
    for first in (-1, 3 * hidden):
        with pytest.raises(_lib.KsError):
            _lib.check(cell._lib.ks_mlps_copy_params_from(one(cell.proj_h._handle), 1, _lib.current_stream(), one(out.data_ptr()), one(out.data_ptr()),
                                                          (ctypes.c_int32 * 1)(first), 0))


@pytest.mark.parametrize("kind", ["gru", "lstm"])
def test_a_given_projected_input_is_checked(kind):
    """Rows too few, rows of another width, another type, gaps between rows, host memory: nothing of this is handed to a launch."""
    from ksim_amd import _lib
    from ksim_amd.recurrent import GRUCell, LSTMCell, run_sequences

    steps, rows, H, G = 3, 5, 128, 3 if kind == "gru" else 4
    rng = np.random.default_rng(0)
    w = [rng.normal(scale=H ** -0.5, size=s) for s in ((G * H, H), (G * H, H), (G * H,))]
    cell = GRUCell(*w, rng.normal(size=H), dtype="f32") if kind == "gru" else LSTMCell(*w, dtype="f32")
    x, fresh = torch.randn(steps, rows, H, device="cuda"), torch.zeros(steps, rows, dtype=torch.uint8, device="cuda")
    carry = [torch.randn(rows, H, device="cuda") for _ in range(1 if kind == "gru" else 2)]

    def call(gi):
        outs = [torch.empty(steps, rows, H, device="cuda") for _ in carry]
        return cell.sequence_call(x, *carry, fresh, *outs, None, gi), outs

    good = cell._input_projection()(x.view(steps * rows, H))
    for bad in (good[:-1], good[:, :-1].contiguous(), good.view(steps, rows, G * H), good.double(), good.half(), torch.cat([good, good], 1)[:, : G * H], good.cpu()):
        with pytest.raises(_lib.KsError):
            call(bad)
    (given, got), (own, want) = call(good), call(None)
    run_sequences([given])
    run_sequences([own])
    assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
def test_training_forward_of_what_cannot_be_trained_is_refused(dtype):
    """An output layer without its training buffers, and a trajectory of no steps: the same answer in both precisions."""
    from ksim_amd import _lib
    from ksim_amd.mlp import MLP
    from ksim_amd.recurrent import GRUCell, RecurrentNetwork

    rng = np.random.default_rng(3)
    w = lambda *s: rng.normal(scale=0.1, size=s)  # noqa: E731

    def net(H):
        return RecurrentNetwork((w(H, 6), w(H)), [GRUCell(w(3 * H, H), w(3 * H, H), w(3 * H), w(H), dtype=dtype)],
                                MLP([w(4, H)], [w(4)], activation="none", dtype=dtype), dtype=dtype)

    def args(T, M, H):
        return torch.randn(T, M, 6, device="cuda"), torch.zeros(1, M, H, device="cuda"), torch.zeros(T, M, dtype=torch.uint8, device="cuda")

    part = net(128)
    part.input_proj.train_init()
    part.cells[0].train_init()
    with pytest.raises(_lib.KsError, match="ks_mlp_train_init"):
        part.train_forward(*args(2, 3, 128))
    whole = net(64)  # a width whose cells step one by one
    whole.train_init()
    with pytest.raises(_lib.KsError):
        whole.train_forward(*args(0, 3, 64))
    assert whole.train_forward(*args(2, 3, 64)).shape == (2, 3, 4)


@pytest.mark.parametrize("kind,dtype,H", [("gru", "bf16", 128), ("gru", "f32", 128), ("gru", "bf16", 64), ("lstm", "f32", 128), ("lstm", "f32", 96)])
def test_weight_gradients_layer_by_layer_are_those_of_one_launch(kind, dtype, H, monkeypatch):
    """Above `LATER_ROWS` rows every layer's gradients are launched when they are due, below it all weight gradients at the end: the same bits, for two
    networks side by side, with cells of the sequence kernels and without."""
    from ksim_amd import recurrent
    from ksim_amd.mlp import MLP
    from ksim_amd.recurrent import GRUCell, LSTMCell, RecurrentNetwork, lockstep

    steps, rows, G = 5, 37, 3 if kind == "gru" else 4
    rng = np.random.default_rng(H)
    w = lambda *s: rng.normal(scale=s[-1] ** -0.5, size=s)  # noqa: E731

    def net(inputs, outputs):
        cells = [GRUCell(w(G * H, H), w(G * H, H), w(G * H), w(H), dtype=dtype) if kind == "gru" else LSTMCell(w(G * H, H), w(G * H, H), w(G * H), dtype=dtype)
                 for _ in range(2)]
        return RecurrentNetwork((w(H, inputs), w(H)), cells, MLP([w(outputs, H)], [w(outputs)], activation="none", dtype=dtype), dtype=dtype)

    nets, passes = [net(43, 40), net(65, 1)], []
    for n in nets:
        n.train_init()
        carry = torch.from_numpy(0.3 * rng.normal(size=(2, 2, rows, H) if kind == "lstm" else (2, rows, H)).astype(np.float32)).cuda()
        obs, d_out = (torch.from_numpy(rng.normal(size=(steps, rows, k)).astype(np.float32)).cuda() for k in (n.in_dim, n.out_dim))
        passes.append((obs, carry, torch.from_numpy((rng.random((steps, rows)) < 0.1).astype(np.uint8)).cuda(), d_out))
    results = []
    for limit in (steps * rows, steps * rows - 1):
        monkeypatch.setattr(recurrent, "LATER_ROWS", limit)
        for n, (obs, carry, fresh, _) in zip(nets, passes):
            n.train_forward(obs, carry, fresh)
        lockstep(*(n.backward_pass(d_out) for n, (_, _, _, d_out) in zip(nets, passes)))
        results.append([g.clone() for n in nets for m in n.networks() for pair in m.parameters(gradients=True) for g in pair])
    assert len(results[0]) == 24 and all(bool(g.any()) for g in results[0])
    assert all(torch.equal(a, b) for a, b in zip(*results))


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
def test_observations_of_one_column_train_whatever_its_stride(dtype):
    """A contiguous array says nothing by the stride of a dimension of one entry: features first, then permuted, is the same rows."""
    from ksim_amd.mlp import MLP
    from ksim_amd.recurrent import GRUCell, RecurrentNetwork

    H, steps, rows = 128, 4, 9
    rng = np.random.default_rng(5)
    w = lambda *s: rng.normal(scale=0.1, size=s)  # noqa: E731
    net = RecurrentNetwork((w(H, 1), w(H)), [GRUCell(w(3 * H, H), w(3 * H, H), w(3 * H), w(H), dtype=dtype)], MLP([w(4, H)], [w(4)], activation="none", dtype=dtype),
                           dtype=dtype)
    net.train_init()
    permuted = torch.randn(1, steps, rows, device="cuda").permute(1, 2, 0)
    assert permuted.is_contiguous() and permuted.stride(2) != 1
    carry, fresh, d_out = torch.zeros(1, rows, H, device="cuda"), torch.zeros(steps, rows, dtype=torch.uint8, device="cuda"), torch.randn(steps, rows, 4, device="cuda")
    results = []
    for obs in (permuted.clone(memory_format=torch.contiguous_format).view(-1).view(steps, rows, 1), permuted):
        out = net.train_forward(obs, carry, fresh)
        net.backward(d_out)
        results.append([out] + [g.clone() for pair in net.input_proj.parameters(gradients=True) for g in pair])
    assert all(torch.equal(a, b) for a, b in zip(*results))


@pytest.mark.parametrize("rows", [3, 1027])
def test_lstm_sequences_take_infinite_and_very_large_operands_as_a_plain_product_does(rows):
    """The products are made of three parts per operand, of which those of an infinity are NaN and those of large values overflow by themselves:
    against the same steps in 64 bits, forward with such weights and initial states, backward with such gradients and weights, four and
    eight rows per workgroup.  Finite entries to 2e-6 (a gate's preactivation to 1e-6 of a sum of 128 terms below 1, the hardware
    exponential and reciprocal beside it), the others in kind."""
    from ksim_amd.recurrent import LSTMCell

    H, Tn = 128, 3
    rng = np.random.default_rng(83)
    for kind in ("ordinary", "infinite state", "large state", "infinite weight", "infinite gradient", "large gradient", "NaN gradient"):
        w = [rng.normal(scale=H ** -0.5, size=s).astype(np.float32) for s in ((4 * H, H), (4 * H, H), (4 * H,))]
        h0, c0 = (0.5 * rng.normal(size=(rows, H)).astype(np.float32) for _ in range(2))
        x, dH = (rng.normal(size=(Tn, rows, H)).astype(np.float32) for _ in range(2))
        if kind == "infinite state":
            h0[rows - 1, 5] = np.inf
        elif kind == "large state":
            h0[0, 7] = -3e37
        elif kind == "infinite weight":
            w[1][3 * H + 9, 11] = -np.inf
        elif kind.endswith("gradient"):
            dH[1, rows - 1, 64] = {"infinite": -np.inf, "large": 1e36, "NaN": np.nan}[kind.split()[0]]
        cell = LSTMCell(*w, dtype="f32")
        cell.train_init()
        z = lambda n: torch.zeros(Tn, rows, n * H, device=DEV)  # noqa: E731
        hs, cs, sv, dg = z(1), z(1), z(7), z(4)
        fresh = torch.zeros(Tn, rows, dtype=torch.uint8, device=DEV)
        cell.sequence_forward(t32(x), t32(h0), t32(c0), fresh, hs, cs, sv)
        wi, wh, b = (torch.from_numpy(a).double() for a in w)
        h, c, want = torch.from_numpy(h0).double(), torch.from_numpy(c0).double(), []
        for t in range(Tn):
            i, f, g, o = (torch.from_numpy(x[t]).double() @ wi.T + b + h @ wh.T).chunk(4, 1)
            i, f, g, o = i.sigmoid(), f.sigmoid(), g.tanh(), o.sigmoid()
            cn = f * c + i * g
            want.append((i, f, g, o, cn.tanh(), c))
            h, c = o * cn.tanh(), cn
            torch.testing.assert_close(hs[t].cpu().double(), h, rtol=2e-6, atol=2e-6, equal_nan=True, msg=lambda m: f"{kind}, step {t}: {m}")
        if "state" in kind or "weight" in kind:
            continue
        cell.sequence_backward(t32(dH), sv, fresh, dg)
        dh = dc = torch.zeros(rows, H, dtype=torch.float64)
        for t in reversed(range(Tn)):
            i, f, g, o, tc, cp = want[t]
            d = torch.from_numpy(dH[t]).double() + dh
            dct = dc + d * o * (1 - tc * tc)
            gates = torch.cat([dct * g * i * (1 - i), dct * cp * f * (1 - f), dct * i * (1 - g * g), d * tc * o * (1 - o)], 1)
            got = dg[t].cpu().double()
            assert torch.equal(got.isnan(), gates.isnan()) and torch.equal(got.isinf(), gates.isinf()), (kind, t)
            scale = gates.abs().nan_to_num(0, 0, 0).amax(1, keepdim=True).clamp_min(1)
            torch.testing.assert_close((got / scale).nan_to_num(0, 0, 0), (gates / scale).nan_to_num(0, 0, 0), rtol=0, atol=4e-6, msg=lambda m: f"{kind}, step {t}: {m}")
            dc, dh = dct * f, gates @ wh


def _largest_error(got, exact, size):
    """in units of 2^-24 of the terms' size, which is what one rounding may cost at most"""
    return float(((got.double() - exact).abs() / size).max() * 2 ** 24)


@pytest.mark.parametrize("terms", [1, 2])
@pytest.mark.parametrize("rows,Tn", [(5, 1), (5, 2), (1030, 1), (1030, 2)])
def test_lstm_recurrent_products_of_few_terms_round_as_often_as_they_have_terms(rows, Tn, terms):
    """States with one or two entries that are not zero, and gate inputs that take the rounded product away again, so that a preactivation is
    what the product was rounded by.  One step and sequences, four and eight rows per workgroup, against 64 bits: an fp32 sum of n terms
    may be off by n times 2^-24 of their size.  Beside it the sums of the smaller parts' products, below 2^-6 of a term, round four times at
    most, 2^-4 of that unit, and the activations' own 2e-6 of a unit slope are 0.06 of it for terms of 512 and more."""
    from ksim_amd import _lib
    from ksim_amd.recurrent import LSTMCell

    H = 128
    rng = np.random.default_rng(7)
    wh = (rng.choice([-1, 1], (4 * H, H)) * rng.uniform(32, 64, (4 * H, H))).astype(np.float32)
    cell = LSTMCell(np.zeros((4 * H, H), np.float32), wh, np.zeros(4 * H, np.float32), dtype="f32")
    cell.train_init()
    h0 = np.zeros((rows, H), np.float32)
    for m in range(rows):
        h0[m, rng.choice(H, terms, replace=False)] = rng.uniform(16, 32, terms)
    exact, size = h0.astype(np.float64) @ wh.T.astype(np.float64), np.abs(h0).astype(np.float64) @ np.abs(wh.T).astype(np.float64)
    gi = np.zeros((Tn, rows, 4 * H), np.float32)
    gi[0] = -exact
    d, z = t32(gi), lambda *s: torch.zeros(*s, device=DEV)  # noqa: E731
    hs, sv, h, c = z(Tn, rows, H), z(Tn, rows, 7 * H), t32(h0), z(rows, H)
    lib = _lib.load()
    _lib.check(lib.ks_lstm_sequence_forward(cell._handle, _lib.current_stream(), Tn, rows, _lib.ptr(d), _lib.ptr(h), _lib.ptr(c), None, _lib.ptr(hs), None,
                                            _lib.ptr(sv)))
    act = sv[0, :, : 4 * H].cpu().double()  # i | f | g | o; i, f and o are sigmoids, g is a tanh
    pre = torch.logit(act)
    pre[:, 2 * H : 3 * H] = torch.atanh(act[:, 2 * H : 3 * H])
    assert _largest_error(pre, torch.from_numpy(exact + gi[0]), torch.from_numpy(size)) <= terms * (1 + 2**-4) + 0.1


@pytest.mark.parametrize("terms", [1, 2])
@pytest.mark.parametrize("rows", [5, 1030])
def test_lstm_gate_gradients_of_few_terms_round_as_often_as_they_have_terms(rows, terms):
    """The same of the backward product: activations that leave the output gate's gradient alone, a quarter of the hidden state's, one or
    two units with a gradient at the last step, and one before it that takes the rounded product away; no activation rounds here."""
    from ksim_amd import _lib
    from ksim_amd.recurrent import LSTMCell

    H, Tn = 128, 2
    rng = np.random.default_rng(8)
    wh = rng.standard_normal((4 * H, H)).astype(np.float32)
    cell = LSTMCell(np.zeros((4 * H, H), np.float32), wh, np.zeros(4 * H, np.float32), dtype="f32")
    cell.train_init()
    sv = torch.zeros(Tn, rows, 7, H, device=DEV)
    sv[:, :, 3] = 0.5  # the output gate
    sv[:, :, 4] = 1.0  # tanh of the cell state: nothing reaches that
    dH = np.zeros((Tn, rows, H), np.float32)
    for m in range(rows):
        dH[1, m, rng.choice(H, terms, replace=False)] = rng.standard_normal(terms)
    gate, w = 0.25 * dH[1].astype(np.float64), wh[3 * H :].astype(np.float64)
    exact, size = gate @ w, np.abs(gate) @ np.abs(w)
    dH[0] = -exact
    d_g = torch.zeros(Tn, rows, 4 * H, device=DEV)
    lib, d = _lib.load(), t32(dH)
    _lib.check(lib.ks_lstm_sequence_backward(cell._handle, _lib.current_stream(), Tn, rows, _lib.ptr(d), _lib.ptr(sv), None, _lib.ptr(d_g), None, None))
    assert _largest_error(4 * d_g[0, :, 3 * H :].cpu(), torch.from_numpy(exact + dH[0]), torch.from_numpy(size)) <= terms * (1 + 2**-4)


@pytest.mark.parametrize("rows", [5, 1030])
def test_a_row_that_is_not_finite_leaves_the_other_rows_bits_alone(rows):
    """An infinite, a NaN and a very large entry in one row's state or gradient: every other row gets the bits that it has without them, in one
    step, in a sequence and in its backward pass, whose workgroups hold sixteen, four and eight rows."""
    from ksim_amd.recurrent import LSTMCell

    H, Tn, bad = 128, 3, rows - 3
    rng = np.random.default_rng(11)
    w = [rng.normal(scale=H ** -0.5, size=s).astype(np.float32) for s in ((4 * H, H), (4 * H, H), (4 * H,))]
    cell = LSTMCell(*w, dtype="f32")
    cell.train_init()
    h0, c0 = (t32(0.5 * rng.normal(size=(rows, H))) for _ in range(2))
    x, dH = (t32(rng.normal(size=(Tn, rows, H))) for _ in range(2))
    fresh = torch.zeros(Tn, rows, dtype=torch.uint8, device=DEV)
    others = torch.arange(rows, device=DEV) != bad

    def run(value):
        z = lambda t, n: torch.zeros(t, rows, n * H, device=DEV)  # noqa: E731
        h, d = h0.clone(), dH.clone()
        if value is not None:
            h[bad, 5] = d[1, bad, 64] = value
        hs, cs, sv, dg, hs1, cs1, sv1 = z(Tn, 1), z(Tn, 1), z(Tn, 7), z(Tn, 4), z(1, 1), z(1, 1), z(1, 7)
        cell.sequence_forward(x, h, c0, fresh, hs, cs, sv)
        cell.sequence_forward(x[:1].contiguous(), h, c0, fresh[:1].contiguous(), hs1, cs1, sv1)
        assert all(torch.equal(a[0].nan_to_num(7.0), b[0].nan_to_num(7.0)) for a, b in ((hs, hs1), (cs, cs1), (sv, sv1))), value  # a step is a sequence of one
        finite = z(Tn, 7)
        cell.sequence_forward(x, h0, c0, fresh, z(Tn, 1), None, finite)
        cell.sequence_backward(d, finite, fresh, dg)
        return [a[:, others] for a in (hs, cs, sv, dg, hs1, cs1, sv1)]

    want = run(None)
    for value in (float("inf"), float("nan"), 3e37):
        assert all(torch.equal(a, b) for a, b in zip(run(value), want)), value


@pytest.mark.parametrize("rows", [5, 1030])
@pytest.mark.parametrize("steps", [1, 3])
def test_an_episode_start_drops_the_recurrent_product_whatever_the_weights(rows, steps):
    """A fresh row's gates are its input projection alone: an infinite recurrent weight, an infinite or NaN state carried over from the old
    episode change nothing in it, as in the gate kernel of the other hidden sizes."""
    from ksim_amd.recurrent import LSTMCell

    H = 128
    rng = np.random.default_rng(17)
    w = [rng.normal(scale=H ** -0.5, size=s).astype(np.float32) for s in ((4 * H, H), (4 * H, H), (4 * H,))]
    h0, c0 = (0.5 * rng.normal(size=(rows, H)).astype(np.float32) for _ in range(2))
    x = rng.normal(size=(steps, rows, H)).astype(np.float32)
    fresh = rng.random((steps, rows)) < 0.5
    results = []
    for value in (None, np.inf, -np.inf, np.nan):
        wh, h = w[1].copy(), h0.copy()
        if value is not None:
            wh[::7, 11] = value
            h[::2, 3] = value
        cell = LSTMCell(w[0], wh, w[2], dtype="f32")
        cell.train_init()
        hs, cs, sv = (torch.zeros(steps, rows, n * H, device=DEV) for n in (1, 1, 7))
        cell.sequence_forward(t32(x), t32(h), t32(c0), torch.from_numpy(fresh).to(DEV, torch.uint8), hs, cs, sv)
        results.append([a[torch.from_numpy(fresh).to(DEV)] for a in (hs, cs, sv)])
    for other in results[1:]:
        assert all(torch.equal(a, b) for a, b in zip(results[0], other))
    g = torch.from_numpy(x[fresh]).double() @ torch.from_numpy(w[0]).double().T + torch.from_numpy(w[2]).double()
    i, _, c, o = g.chunk(4, 1)  # zero states: no share of the forget gate
    want = o.sigmoid() * (i.sigmoid() * c.tanh()).tanh()
    torch.testing.assert_close(results[0][0].cpu().double(), want, rtol=0, atol=2e-6)  # a sum of 128 terms and the hardware's exponentials


@pytest.mark.parametrize("rows,steps", [(19, 1), (19, 2), (1030, 2)])
def test_lstm_states_may_lie_at_any_float(rows, steps):
    """Initial states that are views one float into a buffer, as float addresses allow: the same bits as at aligned ones."""
    from ksim_amd.recurrent import LSTMCell

    H = 128
    rng = np.random.default_rng(23)
    cell = LSTMCell(*(rng.normal(scale=H ** -0.5, size=s) for s in ((4 * H, H), (4 * H, H), (4 * H,))), dtype="f32")
    h0, c0, x = (t32(rng.normal(size=s)) for s in ((rows, H), (rows, H), (steps, rows, H)))
    fresh = torch.zeros(steps, rows, dtype=torch.uint8, device=DEV)
    results = []
    for shift in (0, 1):
        h, c, hs, cs = (torch.zeros(n * rows * H + 1, device=DEV)[shift : shift + n * rows * H].view(n, rows, H) for n in (1, 1, steps, steps))
        h.copy_(h0[None])
        c.copy_(c0[None])
        cell.sequence_forward(x, h[0], c[0], fresh, hs, cs, None)
        results.append((hs.clone(), cs.clone()))
    assert all(torch.equal(a, b) for a, b in zip(*results))
