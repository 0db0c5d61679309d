"""The surrogate's HIP kernels against the FP64 oracle (oracle/surrogate.py,
pinned by finite differences on the CPU): forward win rates, every
parameter tensor's gradient, the Adam update, checkpoint round trips,
training progress, and the gain over plain playouts.

Layer by layer, each kernel is fed the GPU's own BF16 maps and compared
with the oracle's layer function on the same values: conv outputs and
gradient maps agree to one BF16 rounding step (relative 2^-7) on all but
0.1% of elements, FP32 gradients and head values to 1e-3 relative.

End to end, rounding flips cascade through 13 BF16 layers (on the CPU, the
oracle's own BF16 emulation moves by up to 0.5% per gradient tensor for
these parameters when only its accumulation precision changes), so the
whole-network bars are: win rates within 1e-2 of the BF16-emulating oracle
and 3e-2 of the exact one, per-tensor gradient error below 5% and
whole-vector cosine >= 0.999 against the BF16 oracle, >= 0.995 against the
exact one."""
import os

import numpy as np
import pytest

from oracle import surrogate as orc
from leela_amd import positions
from leela_amd.surrogate import Surrogate, LeafEvaluator, train

pytestmark = pytest.mark.gpu


def _random_params(seed):
    """Every tensor drawn nonzero (the library starts the residual blocks'
    second convs and the output layer at zero, which would leave parts of
    the gradient identically zero), scaled so that the ELU stack stays
    moderate and tanh unsaturated (|t| < 0.5 on generator positions)."""
    rng = np.random.default_rng(seed)
    flat = np.zeros(orc.num_params(), np.float32)
    for name, shape, off in orc.layout():
        n = int(np.prod(shape))
        if name.startswith("W"):
            std = 0.7 * np.sqrt(2.0 / (shape[1] * 9))
        elif name == "F1":
            std = np.sqrt(2.0 / orc.P)
        elif name == "wh":
            std = 0.125
        elif name == "F2":
            std = 0.02
        else:
            std = 0.05
        flat[off:off + n] = rng.normal(0, std, n)
    return flat


@pytest.fixture(scope="module")
def sur():
    s = Surrogate(0, max_batch=512, seed=3)
    s.set_params(_random_params(3))
    yield s
    s.close()


def test_initialisation_starts_blocks_as_identity():
    s = Surrogate(0, max_batch=8, seed=5)
    try:
        p = orc.unpack(s.params().astype(np.float64))
    finally:
        s.close()
    for layer in range(orc.NCONV):
        zero = layer >= 2 and layer % 2 == 0
        assert (np.abs(p[f"W{layer}"]).max() == 0) == zero, layer
        assert np.abs(p[f"b{layer}"]).max() == 0
    assert np.abs(p["F2"]).max() == 0 and np.abs(p["F1"]).max() > 0


def _value_planes(n, seed0):
    return positions.make_batch(n, seed0=seed0, net=positions.NET_VALUE)


def test_forward_matches_oracle(sur):
    print("surrogate forward: 12 generator positions, seeds 500..", flush=True)
    planes = _value_planes(12, 500)
    flat = sur.params().astype(np.float64)
    win = sur.predict(planes)
    t16, _ = orc.forward(flat, planes, bf16_points=True)
    t64, _ = orc.forward(flat, planes)
    assert np.abs(win - (1 + t16) / 2).max() < 1e-2
    assert np.abs(win - (1 + t64) / 2).max() < 3e-2
    # Batches split across predict calls give the same rows.
    np.testing.assert_array_equal(sur.predict(planes[5:9]), win[5:9])


@pytest.mark.parametrize("n", [1, 3, 256, 257])
def test_forward_is_the_same_in_every_batch_size(n):
    """Batches of up to one board per CU run eight waves a board, larger ones
    four: every output is formed by the same operations in the same order,
    so a board's maps and win rate are the same bits in any batch; and the
    first and last board match the oracle (bar as above)."""
    print(f"surrogate forward: {n} positions, seeds 2500..", flush=True)
    planes = _value_planes(n, 2500)
    s = Surrogate(0, max_batch=300, seed=3)
    try:
        s.set_params(_random_params(3))
        flat = s.params().astype(np.float64)
        more = np.concatenate([planes, _value_planes(300 - n, 9000)])
        want = s.predict(more)[:n]
        maps = [s.read_map(0, l, 300)[:n] for l in (0, 1, 12)]
        np.testing.assert_array_equal(s.predict(planes), want)
        for l, m in zip((0, 1, 12), maps):
            np.testing.assert_array_equal(s.read_map(0, l, n), m)
    finally:
        s.close()
    ends = sorted({0, n - 1})
    t16, _ = orc.forward(flat, planes[ends], bf16_points=True)
    assert np.abs(want[ends] - (1 + t16) / 2).max() < 1e-2


def test_gradients_match_oracle(sur):
    print("surrogate gradients: 6 positions, seeds 700..", flush=True)
    planes = _value_planes(6, 700)
    y = np.random.default_rng(1).uniform(0.1, 0.9, 6).astype(np.float32)
    flat = sur.params().astype(np.float64)
    loss, g = sur.gradients(planes, y)
    t, cache = orc.forward(flat, planes, bf16_points=True)
    lo, go = orc.backward(cache, y)
    assert abs(loss - lo) <= 2e-2 * lo + 1e-6
    for name, shape, off in orc.layout():
        n = int(np.prod(shape))
        a, b = g[off:off + n].astype(np.float64), go[off:off + n]
        nb = np.linalg.norm(b)
        if nb < 1e-9:
            assert np.linalg.norm(a) < 1e-6, name
            continue
        rel = np.linalg.norm(a - b) / nb
        assert rel < 0.05, (name, rel)
    g = g.astype(np.float64)
    assert g @ go / np.linalg.norm(g) / np.linalg.norm(go) >= 0.999
    t0, c0 = orc.forward(flat, planes)
    _, g0 = orc.backward(c0, y)
    cos = g @ g0 / np.linalg.norm(g) / np.linalg.norm(g0)
    assert cos >= 0.995
    # Same inputs, same gradient (fixed-order reductions).
    _, g2 = sur.gradients(planes, y)
    np.testing.assert_array_equal(g, g2)


@pytest.mark.parametrize("k", [1, 10, 19, 25, 129, 1025])
def test_gradient_of_a_batch_is_the_mean_of_its_halves(k):
    """2k boards against their two halves: the factor 1 / n halves exactly, so
    every gradient map is half of the half batch's to the bit (in both wave
    grids of the backward pass, and across its split at 1024 boards), and the
    weight gradients differ by the order of FP32 sums only (runs of boards per
    workgroup, the tail of the last run, and the split). Sums of N = 361 n products by magnitude up to 2k boards:
    N^(1/2) ulps at random, 2^-24 * sqrt(361 * 2050) = 5e-5 of the largest
    sum, taken as 1e-4 of the tensor's maximum."""
    print(f"surrogate gradient: 2 x {k} positions", flush=True)
    planes = _value_planes(2 * k, 40000 + k)
    y = np.random.default_rng(k).uniform(0.1, 0.9, 2 * k).astype(np.float32)
    s = Surrogate(0, max_batch=2 * k, seed=3)
    try:
        s.set_params(_random_params(7))
        loss, g = s.gradients(planes, y)
        s.keep_maps(True)
        _, g2 = s.gradients(planes, y)
        layers = (0, 1, 11, 12)
        maps = [_bf(s.read_map(1, l, 2 * k)) for l in layers]
        la, ga = s.gradients(planes[:k], y[:k])
        halves = [[_bf(s.read_map(1, l, k))] for l in layers]
        lb, gb = s.gradients(planes[k:], y[k:])
        for l, h in zip(layers, halves):
            h.append(_bf(s.read_map(1, l, k)))
    finally:
        s.close()
    for l, m, h in zip(layers, maps, halves):
        half = np.concatenate(h) / 2
        # (A half that is a BF16 subnormal is rounded.)
        normal = np.abs(half) >= 2.0 ** -126
        assert normal.mean() > 0.9, l
        np.testing.assert_array_equal(m[normal], half[normal], err_msg=str(l))
    np.testing.assert_array_equal(g, g2)
    assert abs(loss - (la + lb) / 2) <= 1e-5 * abs(loss)
    want = (ga.astype(np.float64) + gb) / 2
    for name, shape, off in orc.layout():
        n = int(np.prod(shape))
        a, b = g[off:off + n], want[off:off + n]
        assert np.abs(b).max() > 0, name
        np.testing.assert_allclose(a, b, rtol=0, atol=1e-4 * np.abs(b).max(),
                                   err_msg=name)


@pytest.mark.parametrize("n", [1, 257])
def test_activation_is_the_float32_elu(n):
    """With zero weights a conv's pre-activation is its bias, so its map is
    ELU(bias) = expf(bias) - 1 in FP32, rounded once to BF16: to the bit
    what torch forms from its float32 exponential. The biases are values
    whose BF16 result is another one if the exponential is formed as 2 to the
    rounded product with log2 e, which is off by up to an ulp more."""
    import torch
    print(f"surrogate ELU: {n} boards", flush=True)

    def result(e, v):
        return torch.where(v > 0, v, e - 1).bfloat16().view(torch.int16)

    g = torch.Generator(device="cuda").manual_seed(1)
    v = -torch.exp2(torch.rand(1 << 24, generator=g, device="cuda") * 16 - 12)
    want = result(torch.exp(v), v)
    at = (want != result(torch.exp2(v * 1.4426950408889634), v)).nonzero()[:, 0]
    assert len(at) > 0
    plain = torch.tensor([1.5, 0.0, -0.5, -3.0, -20.0, -200.0], device="cuda")
    v = torch.cat([v[at], plain])
    want = result(torch.exp(v), v).cpu().numpy().view(np.uint16)
    v = v.cpu().numpy()
    planes = np.zeros((n, 32, 361), np.uint8)
    free = [0, *range(1, orc.NCONV, 2)]  # convs without a residual
    offs = {name: off for name, _, off in orc.layout()}
    s = Surrogate(0, max_batch=n, seed=3)
    try:
        for k in range(0, min(len(v), 2048), 64 * len(free)):
            idx = (np.arange(64 * len(free)) + k) % len(v)
            flat = np.zeros(orc.num_params(), np.float32)
            for l, i in zip(free, idx.reshape(len(free), 64)):
                flat[offs[f"b{l}"]:offs[f"b{l}"] + 64] = v[i]
            s.set_params(flat)
            s.predict(planes)
            for l, i in zip(free, idx.reshape(len(free), 64)):
                got = s.read_map(0, l, n)
                np.testing.assert_array_equal(
                    got, np.broadcast_to(want[i], got.shape), err_msg=str(l))
    finally:
        s.close()


def test_first_step_of_a_fresh_surrogate():
    """Moments and the weight gradients' zero block are zeroed at creation
    (the moments again by set_params), and the first step on the caller's
    stream waits for it: fresh surrogates that get dirty memory make the same
    first step."""
    import torch
    planes = torch.from_numpy(_value_planes(4, 80)).cuda()
    y = torch.tensor([0.2, 0.9, 0.5, 0.4], device="cuda")
    got = []
    for k in range(5):
        print(f"case: fresh surrogate {k}", flush=True)
        junk = [torch.full((1 << 24,), float("nan"), device="cuda")
                for _ in range(6)]
        torch.cuda.synchronize()
        del junk
        torch.cuda.empty_cache()
        st = torch.cuda.Stream()
        s = Surrogate(0, max_batch=4, seed=3)
        try:
            if k:
                s.set_params(got[0][0])
            start = s.params()
            s.train_step_device(4, planes.data_ptr(), y.data_ptr(), 1e-3,
                                stream=st.cuda_stream)
            st.synchronize()
            got.append((start, s.params()))
        finally:
            s.close()
    for start, after in got[1:]:
        np.testing.assert_array_equal(start, got[0][0])
        np.testing.assert_array_equal(after, got[0][1])
    assert np.isfinite(got[0][1]).all()


def _bf(u16):
    """BF16 bit patterns -> float64."""
    return (u16.astype(np.uint32) << 16).view(np.float32).astype(np.float64)


def _nchw(m):
    return np.ascontiguousarray(m.transpose(0, 2, 1))


def _same_bf16(got, ref, what):
    """Equal up to one BF16 rounding step on all but 0.1% of elements."""
    tol = 2.0 ** -7 * np.abs(ref) + 1e-5 * np.abs(ref).max() + 1e-30
    bad = np.mean(np.abs(got - ref) > tol)
    assert bad <= 1e-3, (what, bad)
    assert np.abs(got - ref).max() <= 2.0 ** -5 * np.abs(ref).max() + 1e-30, what


def test_kernels_layer_by_layer():
    print("surrogate layer by layer: 6 positions, seeds 1500..", flush=True)
    n = 6
    s = Surrogate(0, max_batch=16, seed=11)
    try:
        s.set_params(_random_params(11))
        s.keep_maps(True)
        planes = _value_planes(n, 1500)
        y = np.random.default_rng(3).uniform(0.1, 0.9, n).astype(np.float32)
        loss, g = s.gradients(planes, y)
        p = orc.unpack(s.params().astype(np.float64))
        A = [_nchw(_bf(s.read_map(0, l, n))) for l in range(orc.NCONV)]
        E = [_nchw(_bf(s.read_map(1, l, n))) for l in range(orc.NCONV)]
        sv, fv, tv = (v.astype(np.float64) for v in s.read_head(n))
    finally:
        s.close()
    lay = {name: (off, int(np.prod(shape))) for name, shape, off in orc.layout()}

    def grad(name):
        off, cnt = lay[name]
        return g[off:off + cnt].astype(np.float64)

    def inp(layer):
        if layer == 0:
            return planes.reshape(n, 32, 19, 19).astype(np.float64)
        return A[layer - 1].reshape(n, 64, 19, 19)

    # Forward convs: bias, skip and ELU on the GPU's own input maps.
    for layer in range(orc.NCONV):
        res = A[layer - 2] if layer >= 2 and layer % 2 == 0 else None
        z, _ = orc.conv_pre(inp(layer), orc.bf16(p[f"W{layer}"]),
                            p[f"b{layer}"], res)
        _same_bf16(A[layer], orc.bf16(orc._elu(z)), f"conv {layer}")
    # Head forward and backward from the GPU's last map.
    s_o, f_o, t_o = orc.head_fwd(A[-1], p)
    np.testing.assert_allclose(sv, s_o, rtol=1e-4, atol=1e-5)
    np.testing.assert_allclose(fv, f_o, rtol=1e-4, atol=1e-5)
    np.testing.assert_allclose(tv, t_o, rtol=1e-4, atol=1e-5)
    assert abs(loss - orc.loss_of(tv, y)) <= 1e-5
    gh, ds = orc.head_bwd(A[-1], sv, fv, tv, y, p)
    for name in ("wh", "bh", "F1", "c1", "F2", "c2"):
        ref = gh[name].ravel()
        np.testing.assert_allclose(grad(name), ref, rtol=1e-3,
                                   atol=1e-5 * np.abs(ref).max(), err_msg=name)
    _same_bf16(E[-1], orc.bf16(ds[:, None, :] * p["wh"][None, :, None]
                               * orc._elu_grad(A[-1])), "head map")
    # Backward: weight gradients and gradient maps from the GPU's maps.
    for layer in range(orc.NCONV - 1, -1, -1):
        cin = 32 if layer == 0 else 64
        dW, db = orc.conv_wgrad(E[layer], orc._cols(inp(layer)), cin)
        np.testing.assert_allclose(grad(f"W{layer}"), dW.ravel(), rtol=1e-3,
                                   atol=1e-4 * np.abs(dW).max(),
                                   err_msg=f"W{layer}")
        np.testing.assert_allclose(grad(f"b{layer}"), db, rtol=1e-3,
                                   atol=1e-4 * np.abs(db).max(),
                                   err_msg=f"b{layer}")
        if layer == 0:
            break
        dx = orc.conv_bwd_data(E[layer], orc.bf16(p[f"W{layer}"]))
        if layer % 2 == 1:
            dx = dx + E[layer + 1]
        _same_bf16(E[layer - 1], orc.bf16(dx * orc._elu_grad(A[layer - 1])),
                   f"map {layer - 1}")


def test_adam_step_matches_oracle():
    import torch
    print("surrogate adam: 2 steps on 8 positions", flush=True)
    s = Surrogate(0, max_batch=64, seed=9)
    try:
        s.set_params(_random_params(9))
        planes = _value_planes(8, 900)
        y = np.linspace(0.2, 0.8, 8).astype(np.float32)
        X = torch.from_numpy(planes).cuda()
        Y = torch.from_numpy(y).cuda()
        p = s.params().astype(np.float64)
        m = np.zeros_like(p)
        v = np.zeros_like(p)
        lr = 1e-3
        for step in (1, 2):
            _, g = s.gradients(planes, y)
            loss = s.train_step_device(8, X.data_ptr(), Y.data_ptr(), lr,
                                       stream=torch.cuda.current_stream().cuda_stream)
            assert np.isfinite(loss)
            p, m, v = orc.adam(p, g.astype(np.float64), m, v, step, lr)
            got = s.params()
            assert np.abs(got - p).max() < 1e-6, step
            p = got.astype(np.float64)
        assert s.step == 2
    finally:
        s.close()


def test_checkpoint_resume_is_exact(tmp_path):
    import torch
    print("surrogate checkpoint: 3 steps, save after 2, resume", flush=True)
    planes = _value_planes(32, 1200)
    y = np.random.default_rng(2).uniform(0, 1, 32).astype(np.float32)
    X = torch.from_numpy(planes).cuda()
    Y = torch.from_numpy(y).cuda()
    st = torch.cuda.current_stream().cuda_stream
    a = Surrogate(0, max_batch=32, seed=4)
    b = Surrogate(0, max_batch=32, seed=5)
    try:
        for _ in range(2):
            a.train_step_device(32, X.data_ptr(), Y.data_ptr(), 1e-3, stream=st)
        path = tmp_path / "sg.ckpt"
        a.save(path)
        a.train_step_device(32, X.data_ptr(), Y.data_ptr(), 1e-3, stream=st)
        b.load(path)
        assert b.step == 2
        b.train_step_device(32, X.data_ptr(), Y.data_ptr(), 1e-3, stream=st)
        np.testing.assert_array_equal(a.params(), b.params())
        with open(tmp_path / "bad.ckpt", "wb") as fp:
            fp.write(b"not a checkpoint")
        with pytest.raises(Exception):
            b.load(tmp_path / "bad.ckpt")
    finally:
        a.close()
        b.close()


def test_batch_limits_rejected(sur):
    with pytest.raises(Exception):
        sur.gradients(np.zeros((0, 32, 361), np.uint8), np.zeros(0, np.float32))
    with pytest.raises(Exception):
        sur.predict(np.zeros((2, 32, 360), np.uint8))


def test_training_beats_playouts_at_equal_cost():
    """Gain over the method without a surrogate. Train on 16,384 generator
    positions labelled with 32 playouts each (600 Adam steps of 256, lr
    1e-3 after warm-up); on 1,024 held-out positions, measure the mean
    absolute error against a fresh 256-playout mean. The surrogate must beat
    the constant predictor by 20% and a 16-playout estimate (16x the
    playouts the labels' noise would suggest), and answer faster than those
    16 playouts run on the host threads."""
    import time
    import torch
    print("surrogate training: labels 16384 x 32 playouts", flush=True)
    th = min(16, os.cpu_count() or 1)
    tr_planes, tr_y = positions.value_labels(16384, 30000, 32, 3_000_000,
                                             threads=th)
    ev_planes, ev_y = positions.value_labels(1024, 40000, 256, 4_000_000,
                                             threads=th)
    s = Surrogate(0, max_batch=1024, seed=7)
    try:
        print("surrogate training: 600 steps, batch 256", flush=True)
        losses = train(s, tr_planes, tr_y, steps=600, batch=256, lr=1e-3,
                       seed=1, log_every=100)
        assert losses[-1][1] < 0.8 * losses[0][1]
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        pred = s.predict(ev_planes)
        t_sur = time.perf_counter() - t0
    finally:
        s.close()
    t0 = time.perf_counter()
    _, est16 = positions.value_labels(1024, 40000, 16, 5_000_000,
                                      threads=th, planes=False)
    t_po = time.perf_counter() - t0
    mae_sur = float(np.mean(np.abs(pred - ev_y)))
    mae_const = float(np.mean(np.abs(tr_y.mean() - ev_y)))
    mae_16 = float(np.mean(np.abs(est16 - ev_y)))
    print(f"MAE surrogate {mae_sur:.4f} constant {mae_const:.4f} "
          f"16-playout {mae_16:.4f}; time surrogate {t_sur * 1e3:.1f} ms, "
          f"16 playouts x 1024 positions on {th} threads {t_po * 1e3:.1f} ms",
          flush=True)
    assert mae_sur < 0.8 * mae_const
    assert mae_sur < mae_16
    assert t_sur < t_po


def test_training_on_the_reference_teacher():
    """The same gain test with the reference's own playout policy as the
    teacher (pattern playouts on the GPU, equal to the host's and the
    reference's): 16,384 positions x 32 pattern playouts for training,
    1,024 held-out positions judged against a fresh 256-playout mean of the
    same policy. The surrogate must beat the constant predictor by 20% and
    a 16-playout estimate of that policy."""
    import torch
    from leela_amd.positions import PLAYOUT_PATTERN
    print("surrogate training: labels 16384 x 32 pattern playouts", flush=True)
    tr_planes, tr_y = positions.value_labels_device(
        16384, 30000, 32, 3_000_000, batch=4096, policy=PLAYOUT_PATTERN)
    ev_planes, ev_y = positions.value_labels_device(
        1024, 40000, 256, 4_000_000, batch=1024, policy=PLAYOUT_PATTERN)
    _, est16 = positions.value_labels_device(
        1024, 40000, 16, 5_000_000, batch=1024, planes=False,
        policy=PLAYOUT_PATTERN)
    s = Surrogate(0, max_batch=1024, seed=7)
    try:
        print("surrogate training: 600 steps, batch 256", flush=True)
        losses = train(s, tr_planes, tr_y, steps=600, batch=256, lr=1e-3,
                       seed=1, log_every=100)
        assert losses[-1][1] < 0.8 * losses[0][1]
        pred = s.predict(ev_planes)
        torch.cuda.synchronize()
    finally:
        s.close()
    mae_sur = float(np.mean(np.abs(pred - ev_y)))
    mae_const = float(np.mean(np.abs(tr_y.mean() - ev_y)))
    mae_16 = float(np.mean(np.abs(est16 - ev_y)))
    print(f"pattern teacher: MAE surrogate {mae_sur:.4f} constant "
          f"{mae_const:.4f} 16-playout {mae_16:.4f}", flush=True)
    assert mae_sur < 0.8 * mae_const
    assert mae_sur < mae_16


def test_config4_at_full_scale(capsys):
    """The surrogate workload at its stated scale, through the training CLI:
    200,000 generator positions (seeds 10000.., move counts 0..250) labelled
    with the mean of 256 GPU playouts each, Adam at lr 1e-3 with batch 512
    (8 epochs), inference at batch 4096, and the error judged as MAE against
    a fresh 256-playout mean on 4,096 held-out positions. The surrogate
    must beat a 64-playout estimate and the constant predictor, and answer
    at batch 4096 faster than the host threads produce 256-playout
    estimates."""
    import json
    from leela_amd import train_surrogate
    print("config 4: 200000 x 256 GPU playouts, 8 epochs of batch 512",
          flush=True)
    rc = train_surrogate.main(["--n", "200000", "--seed0", "10000",
                               "--playouts", "256", "--epochs", "8",
                               "--batch", "512", "--lr", "1e-3",
                               "--eval-n", "4096", "--eval-playouts", "256",
                               "--infer-batch", "4096", "--log-every",
                               "1000"])
    assert rc == 0
    out = json.loads(capsys.readouterr().out.strip().splitlines()[-1])
    with capsys.disabled():
        print(f"config 4: MAE surrogate {out['mae_surrogate']:.4f}, "
              f"64 playouts {out['mae_64_playouts']:.4f}, constant "
              f"{out['mae_constant']:.4f}; data {out['data_seconds']} s, "
              f"training {out['train_seconds']} s, inference "
              f"{out['infer_positions_per_s']:.0f} positions/s at 4096")
    assert out["mae_surrogate"] < out["mae_64_playouts"]
    assert out["mae_surrogate"] < 0.8 * out["mae_constant"]
    assert out["infer_positions_per_s"] > out["playout_estimates_per_s"]
