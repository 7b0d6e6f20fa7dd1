"""GPU kernels at the edges of the sizes they serve (tile and wave remainders,
the smallest and largest of a range), against the CPU oracle.

Tolerance of a training step: rel 1e-4 / abs 1e-5 per element after a few SGD
steps, as the parity tests state it for fp32.
"""
import numpy as np
import pytest

from tests.oracle_lib import load_oracle
from tests.test_gpu_parity import _launch_labels, assert_params_close, close_enough, run_steps, say
from tests.test_planner import forms
from volta_amd import DeviceArray, data, load_hip
from volta_amd.abi import STATUS_BAD_ARGUMENT, STATUS_NONFINITE_LOSS, MlpSpec, Trainer

pytestmark = pytest.mark.gpu


def against_oracle(spec, B, lr=0.01, steps=3, seed=7):
    """Losses and parameters after `steps` steps on fresh batches, HIP against oracle."""
    ws, bs = data.he_uniform(seed, spec.sizes)
    batches = [data.batch(seed + 1 + s, spec.sizes, B, spec.loss) for s in range(steps)]
    lh, wh, bh, st = run_steps(load_hip(), spec, B, ws, bs, batches, lr, steps)
    lo, wo, bo, _ = run_steps(load_oracle(), spec, B, ws, bs, batches, lr, steps)
    assert st == 0, f"status {st}"
    ok, mx, _ = close_enough(lh, lo)
    assert ok, f"losses differ, max abs {mx:.3e}\n hip={lh}\n ora={lo}"
    assert_params_close(wh, bh, wo, bo, spec.text())


def resumed_run(lib, spec, B, lr, steps=3, seed=7):
    """Losses, parameters and optimizer state after `steps` steps from an optimizer state 1000 steps old:
    first moments of about 1e-3, second ones of about 1e-6 (Adagrad: 1e-4).  A weight moves by about lr a
    step, whatever its gradient, and by an error of a gradient e by about 100 lr e."""
    ws, bs = data.he_uniform(seed, spec.sizes)
    t = Trainer(lib, spec, B)
    t.set_all_params(ws, bs)
    rng, parts = np.random.default_rng(seed), []
    for a in [x for pair in zip(ws, bs) for x in pair]:
        parts.append((1e-3 * rng.standard_normal(a.size), (1e-4 if spec.optimizer == "adagrad" else 1e-6) *
                      (0.5 + rng.random(a.size))))
    state = []
    for i in range(0, len(parts), 2):  # per layer: the moments of W and b, then their second moments
        if spec.optimizer in ("adam", "adamw"):
            state += [parts[i][0], parts[i + 1][0]]
        if spec.optimizer != "sgd":
            state += [parts[i][1], parts[i + 1][1]]
    if state:
        t.set_state(np.concatenate(state).astype(np.float32), 1000)
    losses = []
    for s in range(steps):
        t.step(*data.batch(seed + 1 + s, spec.sizes, B, spec.loss), lr)
        losses.append(t.loss())
    out = losses, *t.get_params(), t.get_state()[0]
    assert t.status() == 0
    t.close()
    return out


def resumed_against_oracle(spec, B, lr=1e-3, steps=3):
    """A resumed run, HIP against oracle: the state within rel 1e-4 and 1e-4 of its rms (what a step adds to it is
    a gradient's share, which differs by some 1e-6 of the gradients' rms)."""
    lh, wh, bh, sh = resumed_run(load_hip(), spec, B, lr, steps)
    lo, wo, bo, so = resumed_run(load_oracle(), spec, B, lr, steps)
    ok, mx, _ = close_enough(lh, lo)
    assert ok, f"losses differ, max abs {mx:.3e}\n hip={lh}\n ora={lo}"
    assert_params_close(wh, bh, wo, bo, spec.text())
    pos = 0
    for r, c in spec.shapes() if so.size else []:
        for n in (r * c, c) * (so.size // sum(r * c + c for r, c in spec.shapes())):
            a, b = sh[pos:pos + n], so[pos:pos + n]
            ok, mx, bad = close_enough(a, b, 1e-4, 1e-4 * float(np.sqrt(np.mean(b.astype(np.float64) ** 2))))
            assert ok, f"{spec.text()}: state at {pos}: {bad} of {n} differ, max abs {mx:.3e}"
            pos += n


# Stand-alone loss heads (more than 64 outputs): one wave per row, rows of up
# to 64, 128, 256 and 1024 columns in registers and longer ones read again;
# four rows per block, several rows per wave above 4096 rows.
@pytest.mark.parametrize("loss,C,B", [("ce", c, b) for c in (65, 128, 129, 1024, 1025) for b in (1, 5)] +
                         [("ce", 100, 4099), ("ce", 257, 66), ("mse", 65, 1), ("mse", 100, 41), ("mse", 67, 4099)])
def test_wide_loss_head(loss, C, B):
    say(f"wide loss head {loss} C={C} B={B}")
    against_oracle(MlpSpec([9, 12, C], "tanh", "sgd", loss), B)


def test_wide_loss_head_special_values():
    """A label outside the classes and an infinite logit: the loss is NaN, the
    label is reported, and the other rows' gradients are what they are without it."""
    say("wide loss head special values")
    lib, C, B = load_hip(), 100, 8
    spec = MlpSpec([4, C], "relu", "sgd", "ce")
    ws, bs = data.he_uniform(1, spec.sizes)
    X, Y = data.batch(2, spec.sizes, B, "ce")
    bad = Y.copy()
    bad[3] = C
    got = []
    for y in (Y, bad):
        t = Trainer(lib, spec, B)
        t.set_all_params(ws, bs)
        dx, dy = DeviceArray(X), DeviceArray(y)
        assert t.step_device(dx.ptr, dy.ptr, 0.0) == 0
        got.append((t.debug_buffer(1, 0).reshape(B, C), t.loss(), t.status()))
        t.close()
    (d0, l0, s0), (d1, l1, s1) = got
    assert s0 == 0 and np.isfinite(l0)
    assert s1 == STATUS_BAD_ARGUMENT | STATUS_NONFINITE_LOSS and np.isnan(l1)
    np.testing.assert_array_equal(np.delete(d0, 3, 0), np.delete(d1, 3, 0))
    X[2, 0] = np.inf
    t = Trainer(lib, spec, B)
    t.set_all_params(ws, bs)
    t.step(X, Y, 0.0)
    assert np.isnan(t.loss()) and t.status() == STATUS_NONFINITE_LOSS
    np.testing.assert_array_equal(np.delete(t.debug_buffer(1, 0).reshape(B, C), 2, 0), np.delete(d0, 2, 0))
    t.close()


# The step's inputs: a host-fed step reads them from a ring of pinned slots (or
# one slot and a copy engine above 1 MiB), a device-fed one from any 4-byte
# aligned address.  Both leave the resident batch and the training as a step on
# the resident batch does, over more steps than the ring has slots.
@pytest.mark.parametrize("L0,B,Ln,loss", [(5, 3, 3, "mse"), (1, 1, 1, "mse"), (7, 33, 10, "ce"), (64, 64, 70, "mse"),
                                          (400, 650, 5, "ce"), (400, 700, 5, "ce"), (401, 701, 1, "mse")])
def test_step_inputs(L0, B, Ln, loss):
    say(f"step inputs L0={L0} B={B} {loss}")
    lib, steps = load_hip(), 7
    spec = MlpSpec([L0, 8, Ln], "tanh", "sgd", loss)
    ws, bs = data.he_uniform(3, spec.sizes)
    batches = [data.batch(40 + s, spec.sizes, B, loss) for s in range(steps)]
    X = np.concatenate([np.zeros(1, np.float32)] + [b[0].ravel() for b in batches])  # every step's X is misaligned
    Y = np.concatenate([np.zeros(1, batches[0][1].dtype)] + [b[1].ravel() for b in batches])
    dx, dy = DeviceArray(X), DeviceArray(Y)
    got = []
    for feed in ("host", "device", "resident"):
        t = Trainer(lib, spec, B)
        t.set_all_params(ws, bs)
        xb, yb = t.batch_buffers()
        for s, (x, y) in enumerate(batches):
            px, py = dx.ptr + 4 + 4 * s * x.size, dy.ptr + 4 + 4 * s * y.size
            if feed == "host":
                x, y = x.copy(), y.copy()
                t.step(x, y, 0.05)
                x.fill(np.nan)  # the caller's arrays are its own again
                y.fill(0)
            elif feed == "device":
                assert t.step_device(px, py, 0.05) == 0
            else:
                assert t.sync() == 0
                assert lib.lib.volta_hip_copy(xb, px, 4 * x.size, 3) == 0
                assert lib.lib.volta_hip_copy(yb, py, 4 * y.size, 3) == 0
                assert t.step_device(xb, yb, 0.05) == 0
        np.testing.assert_array_equal(t.debug_buffer(0, 0), batches[-1][0].ravel())
        got.append((t.loss(), *t.get_params()))
        assert t.status() == 0
        t.close()
    for other in got[1:]:
        assert got[0][0] == other[0]
        for a, b in zip(got[0][1] + got[0][2], other[1] + other[2]):
            np.testing.assert_array_equal(a, b)


# The output layer of up to 64 columns on 16-row strips (one, two and four
# column tiles; strips, K ranges and dX columns with remainders; the strips'
# loss by ticket, by the dW group and by the outer-product dX launch).
@pytest.mark.parametrize("loss,K,N,B", [("ce", 19, 10, 1), ("mse", 1, 2, 17), ("mse", 130, 4, 16), ("ce", 1088, 16, 33),
                                        ("ce", 300, 17, 5), ("mse", 64, 33, 40), ("ce", 129, 64, 256),
                                        ("ce", 3100, 10, 256), ("mse", 50, 3, 257), ("ce", 67, 16, 1025),
                                        ("ce", 48, 40, 513), ("mse", 36, 1, 300)])
@pytest.mark.parametrize("extras", [False, True])
def test_output_strips(loss, K, N, B, extras):
    say(f"output strips {loss} K={K} N={N} B={B} extras={extras}")
    kw = dict(layernorm=True, clip_grad=0.5) if extras else {}
    against_oracle(MlpSpec([8, K, N], "tanh", "sgd", loss, **kw), B)


# Its route: strips, or for 17 to 64 columns and a long K (more than 192 k a
# wave up to 256 rows, from 512 on up to 1024) the product and a loss launch, at
# both sides of each bound.
@pytest.mark.parametrize("loss,K,N,B,strips", [
    ("ce", 1543, 17, 33, True), ("ce", 1544, 17, 33, False), ("mse", 1545, 32, 1, False), ("ce", 771, 33, 256, True),
    ("ce", 772, 33, 256, False), ("mse", 4096, 64, 16, False), ("ce", 2047, 33, 257, True), ("ce", 2048, 64, 257, False),
    ("mse", 2049, 40, 1024, False), ("ce", 2049, 40, 1025, True), ("ce", 4096, 16, 64, True), ("mse", 2050, 16, 300, True)])
def test_output_layer_route(loss, K, N, B, strips):
    say(f"output layer route {loss} K={K} N={N} B={B}")
    spec = MlpSpec([8, K, N], "tanh", "sgd", loss)
    labels = _launch_labels({}, spec, B)
    assert any(x.startswith("fwd1+loss") for x in labels) == strips, labels
    assert ("loss" in labels) == (not strips), labels
    against_oracle(spec, B, steps=2)


# The runtime optimizer's two access widths (whole and partial chunks, aligned
# and misaligned tensors) and its two ways of passing pointers (64 tensors in
# the arguments, more in a table): bit for bit the oracle, as its other tests.
@pytest.mark.parametrize("kind", ["sgd", "adam", "rmsprop", "lars"])
@pytest.mark.parametrize("n", [3, 64, 65])
def test_runtime_optimizer_widths(kind, n):
    from volta_amd.backend import RtOptimizer, config

    say(f"runtime optimizer {kind} n={n}")
    lib, ora = load_hip(), load_oracle()
    counts = [(1023, 1024, 1025, 2048, 5)[i % 5] + (4096 if i == 1 else 0) for i in range(n)]
    rng = np.random.default_rng(n)
    ps = [rng.standard_normal(c + 1).astype(np.float32) for c in counts]
    gs = [rng.standard_normal(c + 1).astype(np.float32) for c in counts]
    dp, dg = [DeviceArray(p) for p in ps], [DeviceArray(g) for g in gs]
    shift = [i % 3 == 2 for i in range(n)]  # misaligned parameter
    gshift = [i % 4 == 3 for i in range(n)]
    hp = [p.copy() for p in ps]
    hip_opt, ora_opt = RtOptimizer(lib.lib, counts), RtOptimizer(ora.lib, counts)
    cfg = config(kind, 0.01, weight_decay=0.01, momentum=0.9)
    for _ in range(3):
        hip_opt.apply(cfg, [d.ptr + 4 * s for d, s in zip(dp, shift)], [d.ptr + 4 * s for d, s in zip(dg, gshift)])
        ora_opt.apply(cfg, [p.ctypes.data + 4 * s for p, s in zip(hp, shift)],
                      [g.ctypes.data + 4 * s for g, s in zip(gs, gshift)])
    for d, p in zip(dp, hp):
        if kind == "lars":  # its norms are a tree, the oracle's sequential: rounding of the local rate
            np.testing.assert_allclose(d.numpy(), p, rtol=1e-5, atol=1e-6)
        else:
            np.testing.assert_array_equal(d.numpy(), p)


# Large states, on loads past the caches and, where a call writes more than
# 352 MiB, on 4-byte accesses: bit for bit the oracle.
@pytest.mark.parametrize("kind,count", [("adam", 26_000_003), ("adam", 31_500_001), ("adagrad", 47_000_001)])
def test_runtime_optimizer_large(kind, count):
    from volta_amd.backend import RtOptimizer, config

    say(f"runtime optimizer {kind} count={count}")
    rng = np.random.default_rng(count)
    p, g = rng.standard_normal(count, np.float32), rng.standard_normal(count, np.float32)
    dp, dg = DeviceArray(p), DeviceArray(g)
    cfg = config(kind, 0.01, weight_decay=0.01)
    RtOptimizer(load_hip().lib, [count]).apply(cfg, [dp.ptr], [dg.ptr])
    RtOptimizer(load_oracle().lib, [count]).apply(cfg, [p.ctypes.data], [g.ctypes.data])
    np.testing.assert_array_equal(dp.numpy(), p)


# Host-fed inference through pinned memory, and above 1 MiB through copies:
# the rows of one call agree with a training handle's forward on the oracle.
@pytest.mark.parametrize("L0,Ln,rows", [(5, 3, 1), (300, 1, 873), (300, 1, 874), (16, 300, 873), (16, 300, 875), (7, 2, 2050)])
def test_host_inference(L0, Ln, rows):
    say(f"host inference {L0} {Ln} rows={rows}")
    spec = MlpSpec([L0, 24, Ln], "relu", "sgd")
    ws, bs = data.he_uniform(4, spec.sizes)
    X = data.normal(9, (rows, L0))
    out = []
    for lib in (load_hip(), load_oracle()):
        t = Trainer(lib, spec, 1024)
        t.set_all_params(ws, bs)
        t.infer(X[: rows // 2 + 1])
        out.append(t.infer(X))
        t.close()
    np.testing.assert_allclose(out[0], out[1], rtol=1e-4, atol=1e-5)


# Sizes of no particular multiple through the small-K dW tiles (rows of 1 to 5
# elements, one past a tile, several 64-k slices), the small-M tile's 16-byte
# loads moved back inside their rows (K of 1 to 5 and remainders of a wave's
# range) and the 64x64 tiles' (larger batches).
@pytest.mark.parametrize("sizes,B", [([1, 2, 3, 4], 1), ([3, 5, 2, 5], 2), ([5, 33, 31, 6], 65), ([4, 65, 64, 7], 64),
                                     ([63, 130, 1, 9, 2], 17), ([257, 18, 515, 3], 256), ([70, 1025, 34, 1], 130),
                                     ([13, 397, 250, 101, 7], 77), ([301, 703, 66, 2], 300), ([530, 1030, 67], 515),
                                     ([2, 771, 3, 770, 5], 641)])
@pytest.mark.parametrize("opt", ["sgd", "adam", "adamw", "adagrad"])
def test_ragged_layers(sizes, B, opt):
    say(f"ragged layers {sizes} B={B} {opt}")
    spec = MlpSpec(sizes, "tanh", opt)
    if opt == "sgd":
        against_oracle(spec, B, lr=0.02)
    else:
        resumed_against_oracle(spec, B)


# The 128x64 direct-to-LDS tile (a grid of a tile per CU, sizes of any
# multiple): integer operands are exact in every order; last stages of 1 to 32
# k, 16- and 4-byte loads.
@pytest.mark.parametrize("layout,M,N,K", [(layout, *s) for layout in (0, 1) for s in (
    (2048, 1024, 128), (1925, 1003, 131), (2044, 1020, 160), (1921, 961, 161), (1001, 1985, 255), (1900, 1050, 289))] +
    # (a dW with K <= 256 is the small-K tile's)
    [(2, *s) for s in ((2048, 1024, 288), (1925, 1003, 257), (2044, 1020, 321), (1921, 961, 319), (1001, 1985, 300),
                       (1900, 1050, 289), (1896, 1048, 320))])
def test_mid_tile_integer_exact(M, N, K, layout):
    """Grids of 256 and of 255 tiles (the tile order over the XCDs with a remainder)."""
    say(f"mid tile {M}x{N}x{K} layout {layout}")
    contig = (M if layout == 2 else K, K if layout == 1 else N)
    assert forms(layout, M, N, K, vec=all(c % 4 == 0 for c in contig)) == (True, False)
    rng = np.random.default_rng(M + layout)
    A = rng.integers(-4, 5, (M, K)).astype(np.float32)
    B = rng.integers(-4, 5, (K, N)).astype(np.float32)
    dA = DeviceArray(np.ascontiguousarray(A.T) if layout == 2 else A)
    dB = DeviceArray(np.ascontiguousarray(B.T) if layout == 1 else B)
    dC = DeviceArray(np.zeros((M, N), np.float32))
    lib = load_hip()
    assert lib.lib.volta_hip_gemm(layout, dA.ptr, dB.ptr, dC.ptr, M, N, K, -1, 0) == 0, lib.last_error()
    np.testing.assert_array_equal(dC.numpy(), A @ B)


@pytest.mark.parametrize("sizes,B,act", [([132, 1992, 1004, 2], 2000, "gelu"), ([131, 1990, 1001, 3], 1999, "relu")])
def test_mid_tile_step(sizes, B, act):
    """Its three epilogues in a training step (products of 256 and 512 tiles)."""
    say(f"mid tile step {sizes} B={B}")
    against_oracle(MlpSpec(sizes, act, "sgd"), B, lr=0.02, steps=2)


@pytest.mark.parametrize("sizes,opt", [([132, 1992, 1004, 2], "adamw"), ([131, 1990, 1001, 3], "adam"),
                                       ([131, 1990, 1001, 3], "adagrad")])
def test_mid_tile_optimizers(sizes, opt):
    """Its dW epilogue on a resumed optimizer state."""
    say(f"mid tile optimizers {sizes} {opt}")
    assert forms(2, *sizes[1:3], 2000, vec=sizes[1] % 4 == 0)[0]
    resumed_against_oracle(MlpSpec(sizes, "tanh", opt), 2000, steps=2)


# The codegen extras' backward launch (rows beside 64-column blocks) and the
# launch that ends their first phase (clip sums, biases, gamma and beta), alone
# and together, over several steps of the dropout stream.
@pytest.mark.parametrize("extras", [dict(layernorm=True), dict(dropout_p=0.2), dict(clip_grad=0.3),
                                    dict(layernorm=True, dropout_p=0.3, clip_grad=0.2)])
@pytest.mark.parametrize("sizes,B", [([5, 2, 1], 1), ([9, 64, 65, 3], 33), ([70, 257, 130, 100], 20), ([16, 40, 12], 300)])
def test_extras_launches(sizes, B, extras):
    say(f"extras {sizes} B={B} {extras}")
    against_oracle(MlpSpec(sizes, "tanh", "sgd", **extras), B)


# Nine weight layers with an output of a few columns: every dW in one launch
# (the most products a group holds), also with the codegen extras.
@pytest.mark.parametrize("B", [7, 256])
@pytest.mark.parametrize("extras", [{}, dict(dropout_p=0.2, clip_grad=0.5)])
def test_dw_group_of_nine(B, extras):
    say(f"dW group of nine layers B={B} {extras}")
    spec = MlpSpec([20, 24, 16, 33, 40, 16, 24, 20, 12, 3], "tanh", "sgd", **extras)
    dws = [label for label in _launch_labels({}, spec, B) if label.startswith("dw")]
    assert len(dws) == 1 and dws[0].count("|") == 8, dws
    against_oracle(spec, B)


# dW groups of aligned and ragged products (an output of a few columns, a
# ragged first or middle layer), on 32x32 and 32x64 tiles: bit for bit the
# products launched one by one, each in its own form.
@pytest.mark.parametrize("sizes,B", [([32, 64, 96, 10], 64), ([30, 64, 128, 4], 33), ([64, 33, 32, 8], 256),
                                     ([20, 48, 16, 3], 1), ([132, 260, 68, 2], 130)])
@pytest.mark.parametrize("tile_n", ["32", "64"])
@pytest.mark.parametrize("opt", ["adam", "adagrad"])
def test_dw_group_mixed_forms(monkeypatch, sizes, B, tile_n, opt):
    say(f"mixed dW group {sizes} B={B} tile_n={tile_n} {opt}")
    spec = MlpSpec(sizes, "tanh", opt)
    monkeypatch.setenv("VOLTA_DW_GROUP_TN", tile_n)
    resumed_against_oracle(spec, B)
    _, w0, b0, s0 = resumed_run(load_hip(), spec, B, 1e-3)
    monkeypatch.setenv("VOLTA_NO_PAIR", "1")
    _, w1, b1, s1 = resumed_run(load_hip(), spec, B, 1e-3)
    for a, b in zip(w0 + b0 + [s0], w1 + b1 + [s1]):
        np.testing.assert_array_equal(a, b)


# A handle's staging memory is pinned with the handle: host-fed steps and host
# inference of any row count, in turn, pin nothing and use the same slots (four
# of a ring, two, one above 1 MiB) without disturbing each other.
@pytest.mark.parametrize("L0,B,Ln", [(5, 3, 2), (100, 257, 9), (300, 900, 3), (16, 900, 300)])
def test_staging_is_the_handles(L0, B, Ln):
    say(f"staging L0={L0} B={B} Ln={Ln}")
    lib = load_hip()
    pinned = lib.lib.volta_hip_pinned_allocations
    spec = MlpSpec([L0, 24, Ln], "tanh", "sgd")
    ws, bs = data.he_uniform(5, spec.sizes)
    batches = [data.batch(60 + s, spec.sizes, B, "mse") for s in range(7)]
    X = data.normal(8, (2 * B + 3, L0))
    got = []
    for infer in (False, True):
        t = Trainer(lib, spec, B)
        before = pinned()
        t.set_all_params(ws, bs)
        for s, (x, y) in enumerate(batches):
            t.step(x, y, 0.05)
            if infer:
                t.infer(X[: 1 + s * X.shape[0] // 7])
        out = t.infer(X)
        assert pinned() == before
        got.append((out, t.loss(), *t.get_params()))
        assert t.status() == 0
        t.close()
    (o0, l0, w0, b0), (o1, l1, w1, b1) = got
    assert l0 == l1
    for a, b in zip([o0] + w0 + b0, [o1] + w1 + b1):
        np.testing.assert_array_equal(a, b)
