"""GPU parity of the surrogate network's BF16 MFMA kernels (liblymph_mlp.so)
against the CPU oracle oracle/mlp_ref.py with the same bfloat16 roundings:
forward outputs, loss, every parameter gradient, and the Adam update.  GPU
and oracle differ only by accumulation order (FP32 on the matrix cores,
float64 in the oracle) and by the rare bfloat16 rounding of an activation
that lands on the other side of a tie, hence the tolerances below."""
import sys

import numpy as np
import pytest

from lymph3d_apsc_amd import device_count
from oracle import mlp_ref as R

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if device_count() == 0:
        pytest.skip("no HIP device")


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a, float) - b) / max(np.linalg.norm(b), 1e-300))


# shapes that exercise full and partial 64x64 tiles, k tails, width 8 and the
# split-k path (output layers of 1536 and 38,400 outputs)
SHAPES = [([8, 64, 64, 128], 64), ([8, 72, 136, 40], 24), ([8, 512, 512, 512, 1536], 128),
          ([8, 64, 64, 38400], 32)]


@pytest.mark.parametrize("widths,batch", SHAPES)
def test_forward_loss_and_gradients_match_oracle(widths, batch):
    from lymph3d_apsc_amd.mlp import Mlp
    say(f"[mlp grads] {widths} batch {batch}")
    rng = np.random.default_rng(len(widths) + batch)
    x = rng.standard_normal((batch, widths[0])).astype(np.float32)
    t = rng.standard_normal((batch, widths[-1])).astype(np.float32)
    with Mlp(widths, max_batch=max(batch, 64), seed=3) as net:
        p = net.params().astype(np.float64)
        y_ref, _ = R.forward(p, widths, x, emulate=True)
        y = net.predict(x)
        assert rel(y, y_ref) < 5e-3
        loss, g = net.gradients(x, t)
        loss_ref, g_ref = R.loss_and_grads(p, widths, x, t, emulate=True)
        assert abs(loss - loss_ref) < 1e-3 * loss_ref
        # per layer: weights and biases
        o = 0
        for k, n in zip(widths[:-1], widths[1:]):
            for size in (n * k, n):
                assert rel(g[o:o + size], g_ref[o:o + size]) < 2e-2, (k, n, size)
                o += size


def test_adam_step_matches_oracle_and_training_reduces_loss():
    from lymph3d_apsc_amd.mlp import Mlp
    say("[mlp train]")
    widths, batch = [8, 64, 64, 32], 32
    rng = np.random.default_rng(11)
    x = rng.standard_normal((256, 8)).astype(np.float32)
    A = rng.standard_normal((8, 32)) / 3
    y = np.tanh(x @ A).astype(np.float32)  # smooth target
    with Mlp(widths, max_batch=64, seed=5) as net:
        net.set_data(x, y)
        p0 = net.params().astype(np.float64)
        order = np.arange(batch, dtype=np.int32)
        _, g = net.gradients(x[:batch], y[:batch])
        net.train(order, batch, lr=1e-3)
        p1 = net.params()
        q, _, _ = R.adam(p0, g.astype(np.float64), 0.0, 0.0, 1, 1e-3)
        assert np.allclose(p1, q, rtol=1e-5, atol=1e-7)
        losses = []
        for epoch in range(60):
            order = rng.permutation(256).astype(np.int32)
            losses.append(net.train(order, batch, lr=3e-3).mean())
        assert losses[-1] < 0.1 * losses[0]
        yp = net.predict(x)
        assert rel(yp, y) < 0.25


# networks on the fragment-order kernels (all widths <= 512) at their edges:
# one layer, widths of one tile and of odd tile counts, the widest, batches of
# half a tile, of a tile and a half and of several slabs; 520 takes the GEMMs
EDGES = [([8, 8], 8), ([16, 24], 24), ([8, 16, 8], 16), ([40, 264, 72, 24], 40), ([32, 512, 512, 512], 72),
         ([512, 8, 504, 16], 8), ([24, 136, 392, 88, 40, 512], 264), ([8, 520, 64, 16], 24)]


@pytest.mark.parametrize("widths,batch", EDGES)
def test_narrow_networks_at_tile_edges_match_oracle(widths, batch):
    """Outputs, loss, gradients and one Adam step against the oracle, to the
    tolerances above (bfloat16 operands, 2^-9 per rounding); every row's
    output is the same bits whatever rows come with it (1, 15, 17 and 4200
    rows: the two slab sizes)."""
    from lymph3d_apsc_amd.mlp import Mlp
    say(f"[mlp edges] {widths} batch {batch}")
    rng = np.random.default_rng(sum(widths) + batch)
    x = rng.standard_normal((4200, widths[0])).astype(np.float32)
    t = rng.standard_normal((batch, widths[-1])).astype(np.float32)
    with Mlp(widths, max_batch=batch + 8, seed=4) as net:
        p = net.params().astype(np.float64)
        y = net.predict(x)
        y_ref, _ = R.forward(p, widths, x[:64], emulate=True)
        assert rel(y[:64], y_ref) < 5e-3
        for n in (1, 15, 17):
            assert np.array_equal(net.predict(x[:n]), y[:n])
        loss, g = net.gradients(x[:batch], t)
        loss_ref, g_ref = R.loss_and_grads(p, widths, x[:batch], t, emulate=True)
        assert abs(loss - loss_ref) < 1e-3 * loss_ref
        o = 0
        for k, n in zip(widths[:-1], widths[1:]):
            for size in (n * k, n):
                assert rel(g[o:o + size], g_ref[o:o + size]) < 2e-2, (k, n, size)
                o += size
        net.set_data(x[:batch], t)
        losses = net.train(np.arange(batch, dtype=np.int32), batch, lr=1e-3)
        q, _, _ = R.adam(p, g.astype(np.float64), 0.0, 0.0, 1, 1e-3)
        assert np.allclose(net.params(), q, rtol=1e-5, atol=1e-7)
        assert abs(losses[0] - loss) <= 1e-6 * loss
        # the packed copies follow the master weights: outputs of a network
        # given the updated parameters are the same bits
        with Mlp(widths, max_batch=batch, seed=0) as other:
            other.set_params(net.params())
            assert np.array_equal(other.predict(x[:33]), net.predict(x[:33]))


# a wide output layer behind hidden layers of at most 512: one tile a wave (520),
# 2 x 2 (8000 x 72) and 4 x 4 (16,408 x 264) with remainders both ways, the
# contraction of its input gradient in one, 2, 8 and 17 parts
WIDE = [([8, 16, 520], 8), ([24, 72, 40, 1032], 24), ([8, 512, 8000], 72), ([16, 40, 16408], 264)]


@pytest.mark.parametrize("widths,batch", WIDE)
def test_wide_outputs_at_tile_edges_match_oracle(widths, batch):
    """The checks above; 4200 rows of 16,408 outputs come in several chunks."""
    test_narrow_networks_at_tile_edges_match_oracle(widths, batch)


def test_wide_update_with_streamed_masters_matches_oracle():
    """The checks above with masters and moments of the output layer above 128
    MB (512 x 21,896: remainders in n), where the update streams them."""
    test_narrow_networks_at_tile_edges_match_oracle([8, 512, 21896], 24)


def free_bytes():
    """Free device memory, from the HIP runtime that liblymph_mlp.so is linked to
    (found through its handle; the process may hold another one)."""
    import ctypes as C
    from lymph3d_apsc_amd import mlp
    hip = mlp.lib()
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipDeviceSynchronize() == 0 and hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("widths,n", [([512, 8], 150000), ([1024, 8], 80000), ([8, 16, 1032], 50000)])
def test_predict_keeps_no_device_memory_of_a_large_call(widths, n):
    """300 MB of inputs (both kinds of network) or 200 MB of outputs: at most the
    two buffers of 64 MB and the hidden activations stay with the network, and
    every row's output is the same bits as in calls of part of the rows, on
    either side of the places where the call is split."""
    from lymph3d_apsc_amd.mlp import Mlp
    say(f"[mlp predict memory] {widths} {n} rows")
    x = np.random.default_rng(n).standard_normal((n, widths[0])).astype(np.float32)
    with Mlp(widths, max_batch=64, seed=2) as net:
        net.predict(x[:64])
        before = free_bytes()
        y = net.predict(x)
        assert before - free_bytes() < 150 << 20
        for i in (0, 16000, 32000, 32700, n - 333):
            assert np.array_equal(net.predict(x[i:i + 333]), y[i:i + 333]), i


# inputs on either side of the width from which they are packed ahead of the
# first layer (128), whole and ragged steps of 32 and tiles of 16 rows, one
# layer and several, batches of several thousand rows
@pytest.mark.parametrize("widths,batch", [([128, 24], 8), ([136, 24], 8), ([136, 520, 8], 24), ([264, 16, 8], 40),
                                          ([504, 512], 2056), ([512, 40, 1032], 264)])
def test_wide_inputs_packed_ahead_match_oracle(widths, batch):
    test_narrow_networks_at_tile_edges_match_oracle(widths, batch)


# few weight tiles and a batch of 2048 and more: four pairs of waves share the
# batch, in lots of 128 rows (remainders of 8 rows up to three lots), tiles past
# the widths' ends, up to 256 workgroups of tiles; 2040 rows are one sum
@pytest.mark.parametrize("widths,batch", [([8, 8], 2048), ([72, 40], 2056), ([24, 136, 88, 8], 2424), ([264, 72], 4096),
                                          ([8, 520], 2176), ([512, 512], 2048), ([504, 8, 520, 16], 2056), ([72, 40], 2040)])
def test_updates_over_large_batches_match_oracle(widths, batch):
    test_narrow_networks_at_tile_edges_match_oracle(widths, batch)


# input gradients of a wide layer over so many rows that a GEMM would not split
# them: 4096 outputs and more in 8 parts (the last one a remainder, the last row
# tiles a half block), 4088 in one
@pytest.mark.parametrize("widths,batch", [([8, 512, 4096], 2048), ([8, 504, 4104], 2056), ([8, 512, 4088], 2048)])
def test_wide_input_gradients_over_large_batches_match_oracle(widths, batch):
    test_narrow_networks_at_tile_edges_match_oracle(widths, batch)


def test_predict_in_pieces_of_a_large_batch_gives_the_bits_of_small_calls():
    """4200 rows of 16,408 outputs on a network of that batch: pieces of 2304
    rows (150 MB of outputs in whole groups of 256); the same rows on a network
    of batch 64, in pieces of 1,000 and less."""
    from lymph3d_apsc_amd.mlp import Mlp
    say("[mlp predict pieces]")
    widths = [8, 40, 16408]
    x = np.random.default_rng(9).standard_normal((4200, 8)).astype(np.float32)
    with Mlp(widths, max_batch=4200, seed=6) as net, Mlp(widths, max_batch=64, seed=6) as small:
        y = net.predict(x)
        assert np.isfinite(y).all() and np.abs(y).min(axis=1).max() > 0
        for a in range(0, 4200, 1000):
            assert np.array_equal(small.predict(x[a:a + 1000]), y[a:a + 1000]), a
        y_ref, _ = R.forward(net.params().astype(np.float64), widths, x[2290:2320], emulate=True)
        assert rel(y[2290:2320], y_ref) < 5e-3


@pytest.mark.parametrize("widths,max_batch", [([512, 512, 512], 8), ([24, 512, 488, 512, 40], 24), ([8, 512, 512, 512, 1032], 64),
                                              ([136, 504, 512, 8], 32)])
def test_predictions_of_few_rows_by_layers_give_the_bits_of_the_slab(widths, max_batch):
    """Up to 32 rows (of the batch's whole tiles) of a network with large layers
    go a launch per layer, more rows in slabs: the same bits, also between
    training steps, whose buffers they pass through."""
    from lymph3d_apsc_amd.mlp import Mlp
    say(f"[mlp few rows] {widths} {max_batch}")
    rng = np.random.default_rng(max_batch)
    x = rng.standard_normal((100, widths[0])).astype(np.float32)
    t = rng.standard_normal((100, widths[-1])).astype(np.float32)
    with Mlp(widths, max_batch=max_batch, seed=8) as net, Mlp(widths, max_batch=max_batch, seed=8) as other:
        for m in (net, other):
            m.set_data(x, t)
        for step in range(3):
            y = net.predict(x)
            for n in (1, 7, 8, 16, 17, 31, 32, 33):
                assert np.array_equal(net.predict(x[:n]), y[:n]), n
            y_ref, _ = R.forward(net.params().astype(np.float64), widths, x[:16], emulate=True)
            assert rel(y[:16], y_ref) < 5e-3
            order = rng.integers(0, 100, 8).astype(np.int32)
            assert np.array_equal(net.train(order, 8, 1e-3), other.train(order, 8, 1e-3))
            assert np.array_equal(net.params(), other.params())
