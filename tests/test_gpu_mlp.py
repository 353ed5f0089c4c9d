"""GPU parity of turq_mlp: down(act(gate(x)) * up(x)), the reference's whole MLP (src/models/qwen3.rs:161-167,
src/models/granite_41.rs:151-155), called through the C ABI.

The contract is "the results of turq_qmatmul_gate_up into f32 followed by turq_qmatmul, bit for bit"; both are checked against
the oracle's matmuls on dequantized weights with the oracle's SiLU product in between (bar 1e-3).
"""
import ctypes

import numpy as np
import pytest

from oracle import capi as orc
from oracle import oracle_np as onp
from tests.helpers import Gpu, rel_l2
from tur_amd import capi, synth

pytestmark = pytest.mark.gpu
Q8_0, Q4_K, Q5_K, Q6_K = 8, 12, 13, 14
# the synthetic weights give products of a few hundred at unit activations, and their product would leave the f16 range that the
# second matmul rounds its input to; real MLPs sit far below that
XS = 0.01


@pytest.fixture(scope="module")
def gpu():
    g = Gpu()
    yield g
    g.close()


def f16_round(x):
    return x.astype(np.float16).astype(np.float32)


def expected(dt_gu, dt_dn, x, raw_g, raw_u, raw_d, n_ff, k, n_out, biases=(None, None, None)):
    g = orc.matmul_dequant(dt_gu, x, raw_g, n_ff, k)
    u = orc.matmul_dequant(dt_gu, x, raw_u, n_ff, k)
    if biases[0] is not None:
        g = g + biases[0]
    if biases[1] is not None:
        u = u + biases[1]
    h = onp.silu_mul(g, u)
    y = orc.matmul_dequant(dt_dn, f16_round(h), raw_d, n_out, n_ff)
    return y if biases[2] is None else y + biases[2]


def weights(gpu, dt_gu, dt_dn, n_ff, k, n_out, seed=1, layout=capi.LAYOUT_TILED):
    raws = [synth.random_weight(dt_gu, n_ff, k, seed=seed), synth.random_weight(dt_gu, n_ff, k, seed=seed + 1),
            synth.random_weight(dt_dn, n_out, n_ff, seed=seed + 2)]
    ws = [gpu.upload(dt_gu, n_ff, k, raws[0], layout), gpu.upload(dt_gu, n_ff, k, raws[1], layout),
          gpu.upload(dt_dn, n_out, n_ff, raws[2], layout)]
    return raws, ws


def two_calls(gpu, ws, x, n_ff, k, n_out, x_dtype=capi.ACT_F32, biases=(None, None, None)):
    h = gpu.gate_up(ws[0], ws[1], x, n_ff, k, x_dtype=x_dtype, bias_gate=biases[0], bias_up=biases[1])
    return gpu.qmatmul(ws[2], h, n_out, n_ff, bias=biases[2])


@pytest.mark.parametrize("dt_gu,dt_dn", [(Q4_K, Q4_K), (Q4_K, Q6_K)])
@pytest.mark.parametrize("x_dtype", [capi.ACT_F32, capi.ACT_BF16, capi.ACT_F16])
def test_one_row_equals_the_two_calls(gpu, dt_gu, dt_dn, x_dtype):
    # the MLP of Qwen3-8B at two thirds of its width
    n_ff, k, n_out = 8192, 4096, 4096
    raws, ws = weights(gpu, dt_gu, dt_dn, n_ff, k, n_out, seed=3)
    rng = np.random.default_rng(5)
    biases = tuple(rng.standard_normal(n).astype(np.float32) * 0.1 for n in (n_ff, n_ff, n_out))
    for trial, bs in enumerate([(None, None, None), biases]):
        x = synth.random_activation(1, k, seed=30 + trial) * XS
        if x_dtype == capi.ACT_BF16:
            x = synth.from_bf16_bits(synth.to_bf16_bits(x)).reshape(1, k)
        elif x_dtype == capi.ACT_F16:
            x = f16_round(x)
        launches = []
        y = gpu.mlp(*ws, x, n_ff, k, n_out, x_dtype=x_dtype, biases=bs, launches=launches)
        assert launches == [2], launches
        assert np.isfinite(y).all() and np.abs(y).max() > 0
        assert np.array_equal(y, two_calls(gpu, ws, x, n_ff, k, n_out, x_dtype=x_dtype, biases=bs))
        want = expected(dt_gu, dt_dn, f16_round(x), *raws, n_ff, k, n_out, biases=bs)
        assert rel_l2(y, want) <= 1e-4, rel_l2(y, want)
    for w in ws:
        gpu.release(w)


def test_calls_in_a_row_and_output_dtypes(gpu):
    # different inputs and output types, one call after the other
    n_ff, k, n_out = 8192, 4096, 2048
    raws, ws = weights(gpu, Q4_K, Q4_K, n_ff, k, n_out, seed=7)
    for i in range(6):
        x = synth.random_activation(1, k, seed=50 + i) * (XS * (0.2 + 0.05 * i))
        y_dtype = [capi.ACT_F32, capi.ACT_BF16, capi.ACT_F16][i % 3]
        launches = []
        y = gpu.mlp(*ws, x, n_ff, k, n_out, y_dtype=y_dtype, launches=launches)
        assert launches == [2]
        want = expected(Q4_K, Q4_K, f16_round(x), *raws, n_ff, k, n_out)
        assert rel_l2(y, want) <= (1e-4 if y_dtype == capi.ACT_F32 else 4e-3 if y_dtype == capi.ACT_BF16 else 6e-4)
    for w in ws:
        gpu.release(w)


@pytest.mark.parametrize("dt_gu,dt_dn", [(Q8_0, Q8_0), (Q5_K, Q6_K), (Q6_K, Q6_K), (Q4_K, Q4_K)])
@pytest.mark.parametrize("m", [0, 1, 2, 5, 40])
def test_every_other_case_is_the_two_calls(gpu, dt_gu, dt_dn, m):
    # small or ragged shapes, several rows, every format
    n_ff, k, n_out = 768, 512 + (32 if dt_gu == Q8_0 else 0), 200
    raws, ws = weights(gpu, dt_gu, dt_dn, n_ff, k, n_out, seed=11)
    x = synth.random_activation(m, k, seed=m + 1) * XS
    y = gpu.mlp(*ws, x, n_ff, k, n_out)
    assert y.shape == (m, n_out)
    if m:
        assert np.array_equal(y, two_calls(gpu, ws, x, n_ff, k, n_out))
        want = expected(dt_gu, dt_dn, f16_round(x), *raws, n_ff, k, n_out)
        assert rel_l2(y, want) <= 1e-3, rel_l2(y, want)
    for w in ws:
        gpu.release(w)


def test_host_pointers_and_native_layout(gpu):
    n_ff, k, n_out = 512, 256, 96
    raws, ws = weights(gpu, Q4_K, Q6_K, n_ff, k, n_out, seed=13, layout=capi.LAYOUT_NATIVE)
    x = synth.random_activation(3, k, seed=4) * XS
    want = expected(Q4_K, Q6_K, x, *raws, n_ff, k, n_out)
    assert rel_l2(gpu.mlp(*ws, x, n_ff, k, n_out, mem=capi.MEM_HOST), want) <= 1e-3
    assert rel_l2(gpu.mlp(*ws, x, n_ff, k, n_out), want) <= 1e-3
    for w in ws:
        gpu.release(w)


def test_argument_errors(gpu):
    raws, ws = weights(gpu, Q4_K, Q4_K, 512, 256, 64, seed=17)
    wrong = gpu.upload(Q4_K, 64, 256, synth.random_weight(Q4_K, 64, 256, seed=1), capi.LAYOUT_TILED)
    x = np.zeros((1, 256), np.float32)
    y = np.zeros((1, 64), np.float32)
    L = gpu.L
    call = lambda g, u, d, act=0, mem=capi.MEM_HOST, yt=capi.ACT_F32: L.turq_mlp(gpu.ctx, g, u, d, capi.ptr(x), capi.ACT_F32, 1, 256, capi.ptr(y), yt, 64, None, None, None, act, mem)
    assert call(ws[0], ws[1], ws[2]) == capi.OK
    assert call(None, ws[1], ws[2]) == capi.ERR_INVALID
    assert call(ws[0], ws[1], wrong) == capi.ERR_SHAPE and b"down takes 256 columns" in L.turq_last_error(gpu.ctx)
    assert call(ws[0], wrong, ws[2]) == capi.ERR_SHAPE
    assert call(ws[0], ws[1], ws[2], act=3) == capi.ERR_INVALID
    assert call(ws[0], ws[1], ws[2], mem=7) == capi.ERR_INVALID
    assert call(ws[0], ws[1], ws[2], yt=9) == capi.ERR_DTYPE
    for w in ws + [wrong]:
        gpu.release(w)


def test_inside_a_graph(gpu):
    # three MLP calls back to back (the same input: chained, the synthetic weights would leave the f16 range), captured once and
    # replayed with eager work in between
    n_ff, k, n_out = 8192, 4096, 4096
    raws, ws = weights(gpu, Q4_K, Q6_K, n_ff, k, n_out, seed=19)
    L, ctx = gpu.L, gpu.ctx
    x0 = synth.random_activation(1, k, seed=9) * XS
    bufs = [gpu.dev_buffer(x0)] + [gpu.dev_buffer(np.zeros((1, n_out), np.float32)) for _ in range(3)]

    def chain():
        for i in range(3):
            capi.check(L.turq_mlp(ctx, ws[0], ws[1], ws[2], bufs[0], capi.ACT_F32, 1, k, bufs[i + 1], capi.ACT_F32, n_out, None, None, None,
                                  0, capi.MEM_DEVICE), ctx)

    chain()
    capi.check(L.turq_sync(ctx), ctx)
    eager = gpu.read_back(bufs[3], (1, n_out), np.float32)
    assert np.isfinite(eager).all() and np.abs(eager).max() > 0
    assert rel_l2(eager, expected(Q4_K, Q6_K, f16_round(x0), *raws, n_ff, k, n_out)) <= 1e-4
    capi.check(L.turq_graph_begin(ctx), ctx)
    chain()
    g = ctypes.c_void_p()
    capi.check(L.turq_graph_end(ctx, ctypes.byref(g)), ctx)
    for rep in range(4):
        for b in bufs[1:]:
            capi.check(L.turq_memcpy_h2d(ctx, b, capi.ptr(np.zeros((1, n_out), np.float32)), 4 * n_out), ctx)
        capi.check(L.turq_graph_launch(ctx, g), ctx)
        capi.check(L.turq_sync(ctx), ctx)
        for b in bufs[1:]:
            assert np.array_equal(gpu.read_back(b, (1, n_out), np.float32), eager), rep
        gpu.mlp(*ws, synth.random_activation(1, k, seed=100 + rep) * XS, n_ff, k, n_out)  # eager work between the replays
    L.turq_graph_destroy(g)
    for b in bufs:
        gpu.dev_free(b)
    for w in ws:
        gpu.release(w)


@pytest.mark.parametrize("dt_gu,dt_dn", [(Q4_K, Q6_K), (Q5_K, Q4_K)])
@pytest.mark.parametrize("m", [72, 128, 512])
def test_prompt_chunks(gpu, dt_gu, dt_dn, m):
    """More than 32 rows: gate / up GEMMs into f32 scratch, ONE kernel from the two products to down_proj's fragments (no f16 copy
    of the intermediate, no separate preparation), down_proj's GEMM.  Bit-equal to the two calls, within 1e-3 of the oracle's
    chain; bf16 in and out as a prompt chunk has them, and with biases."""
    n_ff, k, n_out = 3072, 2048, 1536
    raws, ws = weights(gpu, dt_gu, dt_dn, n_ff, k, n_out, seed=23 + m)
    rng = np.random.default_rng(m)
    biases = tuple(rng.standard_normal(n).astype(np.float32) * 0.1 for n in (n_ff, n_ff, n_out))
    x = synth.random_activation(m, k, seed=m, bf16=True) * XS
    x = synth.from_bf16_bits(synth.to_bf16_bits(x)).reshape(m, k)
    for bs in ((None, None, None), biases):
        launches = []
        y = gpu.mlp(*ws, x, n_ff, k, n_out, x_dtype=capi.ACT_BF16, biases=bs, launches=launches)
        assert np.array_equal(y, two_calls(gpu, ws, x, n_ff, k, n_out, x_dtype=capi.ACT_BF16, biases=bs))
        g = orc.matmul_dequant(dt_gu, x, raws[0], n_ff, k) + (0 if bs[0] is None else bs[0])
        u = orc.matmul_dequant(dt_gu, x, raws[1], n_ff, k) + (0 if bs[1] is None else bs[1])
        want = orc.matmul_dequant(dt_dn, onp.silu_mul(g, u).astype(np.float32), raws[2], n_out, n_ff) + (0 if bs[2] is None else bs[2])
        assert rel_l2(y, want) <= 1e-3, rel_l2(y, want)
    yb = gpu.mlp(*ws, x, n_ff, k, n_out, x_dtype=capi.ACT_BF16, y_dtype=capi.ACT_BF16, biases=biases)
    assert np.array_equal(synth.to_bf16_bits(yb).reshape(m, n_out), synth.to_bf16_bits(y).reshape(m, n_out))
    for w in ws:
        gpu.release(w)


def pair_plan(dt_gu, dt_dn, n_ff, k, m):
    """the pair that the call's rules make of gate and up: a tile of the kernel whose waves split the columns, minus the tile form of the other, 0: none"""
    f = capi.lib().turq_mlp_pair_plan
    f.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_int64, ctypes.c_int64, ctypes.c_int64, ctypes.c_int]
    return f(dt_gu, dt_dn, n_ff, k, m, 256)


# pair: minus the tile form of the LDS-tiled kernel (1: 128 x 128, 2: 2 x 2 waves, 3: wide), or 10 r + c: 32 r x 32 c of the other (22 alone and two per CU)
@pytest.mark.parametrize("dt_gu,dt_dn,n_ff,k,m,pair", [
    (Q4_K, Q6_K, 2816, 512, 600, -1), (Q5_K, Q6_K, 2816, 512, 600, -1), (Q6_K, Q6_K, 2816, 512, 600, -1),
    (Q4_K, Q5_K, 3840, 512, 513, -2), (Q4_K, Q6_K, 3840, 512, 513, -2), (Q4_K, Q4_K, 2816, 512, 700, -2), (Q4_K, Q8_0, 2816, 512, 700, -2),
    (Q8_0, Q8_0, 3328, 1024, 2017, -2), (Q8_0, Q4_K, 3328, 1024, 2017, -2),
    (Q4_K, Q8_0, 6400, 256, 545, -3), (Q5_K, Q4_K, 6400, 256, 513, -3), (Q6_K, Q8_0, 6400, 256, 513, -3),
    (Q4_K, Q6_K, 256, 256, 33, 11), (Q4_K, Q6_K, 1280, 1024, 70, 11), (Q8_0, Q8_0, 2304, 1024, 47, 11), (Q6_K, Q6_K, 3072, 1024, 33, 21),
    (Q8_0, Q8_0, 2304, 1024, 174, 22), (Q8_0, Q8_0, 3072, 1024, 300, 22), (Q4_K, Q8_0, 4352, 4096, 190, 22), (Q6_K, Q6_K, 5120, 4096, 77, 32),
    (Q8_0, Q6_K, 5376, 3072, 100, 42), (Q5_K, Q8_0, 12288, 4096, 77, 33)])
def test_prompt_pairs(gpu, dt_gu, dt_dn, n_ff, k, m, pair):
    """Gate and up in one launch that writes down_proj's fragments (blocks of n past the last row, rows past m in the last 32; both fragment orders,
    with the sub-block sums of a Q4_K / Q5_K down_proj): bit-equal to the two calls.  The scales of gate and up differ by 2^9, so that a
    column taken with the other's scale would show."""
    assert pair_plan(dt_gu, dt_dn, n_ff, k, m) == pair
    n_out = 512
    raws = [synth.random_weight(dt_gu, n_ff, k, seed=7), synth.random_weight(dt_gu, n_ff, k, seed=8), synth.random_weight(dt_dn, n_out, n_ff, seed=9)]
    nb = synth.BLOCK_BYTES[dt_gu]
    blocks = raws[1].reshape(-1, nb)
    at = nb - 2 if dt_gu == Q6_K else 0
    for o in (at, at + 2) if dt_gu in (Q4_K, Q5_K) else (at,):
        d = blocks[:, o:o + 2].copy().view(np.float16)
        blocks[:, o:o + 2] = (d * np.float16(2.0 ** -9)).view(np.uint8)
    ws = [gpu.upload(dt, n, kk, raw, capi.LAYOUT_TILED) for dt, n, kk, raw in zip((dt_gu, dt_gu, dt_dn), (n_ff, n_ff, n_out), (k, k, n_ff), raws)]
    rng = np.random.default_rng(m)
    x = rng.standard_normal((m, k)).astype(np.float32) * XS
    for bs in ((None, None, None), tuple(rng.standard_normal(n).astype(np.float32) * 0.1 for n in (n_ff, n_ff, n_out))):
        y = gpu.mlp(*ws, x, n_ff, k, n_out, biases=bs)
        assert np.array_equal(y, two_calls(gpu, ws, x, n_ff, k, n_out, biases=bs))
    for w in ws:
        gpu.release(w)


# the second kernel's pair at the edges of its tiles: columns of one and of several blocks, super-blocks fewer than waves and not a multiple of them, rows
# at and past every tile's height; and with each of its tiles forced
@pytest.mark.parametrize("dt", [Q4_K, Q5_K, Q6_K, Q8_0])
@pytest.mark.parametrize("n_ff,k,m", [(512, 256, 33), (768, 512, 96), (1536, 1280, 65), (512, 256, 129)])
def test_column_pair_edges(gpu, dt, n_ff, k, m):
    import os

    forced = int(os.environ.get("TURQ_GEMM_COLS", "0"))
    pair = pair_plan(dt, Q6_K if dt != Q6_K else Q8_0, n_ff, k, m)
    assert pair == forced if forced else pair > 0
    raws, ws = weights(gpu, dt, Q6_K if dt != Q6_K else Q8_0, n_ff, k, 256, seed=31)
    x = synth.random_activation(m, k, seed=m) * XS
    y = gpu.mlp(*ws, x, n_ff, k, 256)
    assert np.array_equal(y, two_calls(gpu, ws, x, n_ff, k, 256))
    assert rel_l2(y, expected(dt, Q6_K if dt != Q6_K else Q8_0, f16_round(x), *raws, n_ff, k, 256)) <= 1e-3
    for w in ws:
        gpu.release(w)


@pytest.mark.parametrize("tile", ["21", "22", "32", "42", "33"])
def test_column_pair_tiles(tile):
    import os
    import subprocess
    import sys

    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    out = subprocess.run([sys.executable, "-m", "pytest", "-q", "-x", "-m", "gpu", "-k", "test_column_pair_edges", "-p", "no:cacheprovider",
                          os.path.join(root, "tests", "test_gpu_mlp.py")],
                         cwd=root, env=dict(os.environ, TURQ_GEMM_COLS=tile), capture_output=True, text=True, timeout=280)
    assert out.returncode == 0, out.stdout[-3000:] + out.stderr[-1000:]


@pytest.mark.parametrize("dt_gu,dt_dn,n_ff,k,m", [(Q4_K, Q6_K, 2816, 512, 600), (Q5_K, Q4_K, 6400, 256, 513), (Q8_0, Q8_0, 3328, 1024, 2017), (Q4_K, Q6_K, 1280, 1024, 70)])
def test_overflow_inside_a_pair_is_counted(gpu, dt_gu, dt_dn, n_ff, k, m):
    """Rows whose gate or up product, or whose SiLU(gate) * up as f16, is no finite number: the same infinities and NaNs as from the two calls in the same
    rows, the other rows as if they were alone, and the count sees each kind by itself."""
    assert pair_plan(dt_gu, dt_dn, n_ff, k, m) != 0

    def counted():
        n = ctypes.c_uint64()
        capi.check(gpu.L.turq_ctx_nonfinite_count(gpu.ctx, ctypes.byref(n), 1), gpu.ctx)
        return n.value

    _, ws = weights(gpu, dt_gu, dt_dn, n_ff, k, 256, seed=41)
    ok = synth.random_activation(m, k, seed=m) * XS
    counted()
    y_ok = gpu.mlp(*ws, ok, n_ff, k, 256)
    assert np.isfinite(y_ok).all() and counted() == 0
    for row, scale in ((m - 1, 3e3), (5, np.inf), (m // 2, np.nan)):  # finite products too large for f16 together; and none
        x = ok.copy()
        x[row, 3 if not np.isfinite(scale) else slice(None)] = scale if not np.isfinite(scale) else ok[row] * scale
        y = gpu.mlp(*ws, x, n_ff, k, 256)
        assert counted() > 0, scale
        assert not np.isfinite(y[row]).any()
        others = np.arange(m) != row
        assert np.array_equal(y[others], y_ok[others])
        two = two_calls(gpu, ws, x, n_ff, k, 256)
        assert np.array_equal(np.isnan(y[row]), np.isnan(two[row])) and np.array_equal(y[row][~np.isnan(y[row])], two[row][~np.isnan(two[row])])
        counted()
    for w in ws:
        gpu.release(w)


@pytest.mark.parametrize("dt_gu,dt_dn,n_ff,k,m,places", [
    (Q5_K, Q6_K, 512, 512, 48, "aab"), (Q5_K, Q6_K, 2816, 512, 600, "aab"),
    (Q6_K, Q6_K, 512, 512, 48, "aba"), (Q8_0, Q8_0, 512, 512, 40, "abb"), (Q4_K, Q4_K, 512, 512, 64, "aba"), (Q6_K, Q6_K, 512, 512, 48, "aaa")])
def test_one_weight_in_several_places(gpu, dt_gu, dt_dn, n_ff, k, m, places):
    """A prompt chunk's MLP whose gate, up or (square matrices) down is one handle, with block scales of about 2e-5: without the power of two that
    every place's launch multiplies them by, they would lose bits in the f16 subnormals.  Bit-equal to the two calls, each of which looks at
    one place, and near the oracle: 1e-3 of the f16 operands, three times over (gate, up, down)."""
    n_out = k if "a" in places[2] or places[1:] == "bb" else 256
    shapes = [(dt_gu, n_ff, k), (dt_gu, n_ff, k), (dt_dn, n_out, n_ff)]
    made = {}
    for c, (dt, n, kk) in zip(places, shapes):
        if c in made:
            continue
        raw = synth.random_weight(dt, n, kk, seed=ord(c))
        nb = synth.BLOCK_BYTES[dt]
        blocks = raw.reshape(-1, nb)
        at = nb - 2 if dt == Q6_K else 0
        for o in (at, at + 2) if dt in (Q4_K, Q5_K) else (at,):
            blocks[:, o:o + 2] = (blocks[:, o:o + 2].copy().view(np.float16) * np.float16(2.0 ** -9)).view(np.uint8)
        made[c] = (raw, gpu.upload(dt, n, kk, raw, capi.LAYOUT_TILED))
    raws, ws = [made[c][0] for c in places], [made[c][1] for c in places]
    x = synth.random_activation(m, k, seed=m)
    y = gpu.mlp(*ws, x, n_ff, k, n_out)
    assert np.array_equal(y, two_calls(gpu, ws, x, n_ff, k, n_out))
    assert rel_l2(y, expected(dt_gu, dt_dn, f16_round(x), *raws, n_ff, k, n_out)) <= 3e-3
    for raw, w in made.values():
        gpu.release(w)


def test_scratch_of_more_rows_serves_a_capture_of_fewer():
    """540 rows take gate and up as a pair, 500 take the two products through memory: what the first call left behind is enough for a capture of the
    second, in which nothing may be allocated"""
    gpu = Gpu()
    n_ff, k, n_out, big, small = 4096, 1024, 256, 540, 500
    assert pair_plan(Q4_K, Q4_K, n_ff, k, big) != 0 and pair_plan(Q4_K, Q4_K, n_ff, k, small) == 0
    _, ws = weights(gpu, Q4_K, Q4_K, n_ff, k, n_out, seed=43)
    L, ctx = gpu.L, gpu.ctx
    x, y = gpu.dev_buffer(synth.random_activation(big, k, seed=2) * XS), gpu.dev_buffer(np.zeros((big, n_out), np.float32))

    def call(m):
        capi.check(L.turq_mlp(ctx, *ws, x, capi.ACT_F32, m, k, y, capi.ACT_F32, n_out, None, None, None, 0, capi.MEM_DEVICE), ctx)

    call(big)
    capi.check(L.turq_sync(ctx), ctx)
    capi.check(L.turq_graph_begin(ctx), ctx)
    call(small)
    g = ctypes.c_void_p()
    capi.check(L.turq_graph_end(ctx, ctypes.byref(g)), ctx)
    call(small)
    want = gpu.read_back(y, (small, n_out), np.float32)
    for _ in range(3):
        call(big)
        capi.check(L.turq_memcpy_h2d(ctx, y, capi.ptr(np.zeros((small, n_out), np.float32)), 4 * small * n_out), ctx)
        capi.check(L.turq_graph_launch(ctx, g), ctx)
        capi.check(L.turq_sync(ctx), ctx)
        assert np.array_equal(gpu.read_back(y, (small, n_out), np.float32), want)
    L.turq_graph_destroy(g)
    for p in (x, y):
        gpu.dev_free(p)
    for w in ws:
        gpu.release(w)
    gpu.close()
