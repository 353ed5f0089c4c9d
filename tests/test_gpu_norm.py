"""turq_rms_norm against the formula in f64 (candle_nn's RmsNorm as the reference builds it in src/models/layers/norm.rs:52-94:
y = x / sqrt(mean(x^2) + eps) * weight, f32 arithmetic).  The f32 summation order of candle's kernel is not reproduced bit by bit
(parity unpinned at that level: candle-nn is not in the reference tree); the bar is 1e-6 relative, a few f32 ulps."""
import ctypes

import numpy as np
import pytest

from tests.helpers import Gpu, rel_l2
from tur_amd import capi, qlinear, synth
from tur_amd.gguf import write_gguf

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    g = Gpu()
    yield g
    g.close()


def want_norm(x, w, eps):
    x64 = np.asarray(x, np.float64)
    return x64 / np.sqrt((x64 * x64).mean(axis=-1, keepdims=True) + eps) * np.asarray(w, np.float64)


def call(gpu, x, w, eps, x_dtype=capi.ACT_F32, y_dtype=capi.ACT_F32, mem=capi.MEM_HOST, ldx=None, ldy=None):
    m, k = x.shape
    ldx, ldy = ldx or k, ldy or k
    xb = np.zeros((m, ldx), np.float32)
    xb[:, :k] = x
    send = synth.to_bf16_bits(xb).reshape(m, ldx) if x_dtype == capi.ACT_BF16 else xb.astype(np.float16) if x_dtype == capi.ACT_F16 else xb
    ydt = {capi.ACT_F32: np.float32, capi.ACT_BF16: np.uint16, capi.ACT_F16: np.float16}[y_dtype]
    y = np.zeros((m, ldy), ydt)
    w = np.ascontiguousarray(w, np.float32)
    if mem == capi.MEM_DEVICE:
        xd, wd, yd = gpu.dev_buffer(send), gpu.dev_buffer(w), gpu.dev_buffer(y)
        capi.check(gpu.L.turq_rms_norm(gpu.ctx, xd, x_dtype, m, k, ldx, wd, eps, yd, y_dtype, ldy, mem), gpu.ctx)
        y = gpu.read_back(yd, (m, ldy), ydt)
        for p in (xd, wd, yd):
            gpu.dev_free(p)
    else:
        capi.check(gpu.L.turq_rms_norm(gpu.ctx, capi.ptr(send), x_dtype, m, k, ldx, capi.ptr(w), eps, capi.ptr(y), y_dtype, ldy, mem), gpu.ctx)
    if y_dtype == capi.ACT_BF16:
        y = synth.from_bf16_bits(y).reshape(m, ldy)
    return np.asarray(y, np.float32)[:, :k]


@pytest.mark.parametrize("mem", [capi.MEM_HOST, capi.MEM_DEVICE], ids=["host", "device"])
@pytest.mark.parametrize("m,k", [(1, 4096), (5, 1024), (64, 4096), (3, 5), (2, 4100), (7, 12288), (1, 1)])
def test_rms_norm_f32(gpu, m, k, mem):
    rng = np.random.default_rng(m * 1000 + k)
    x = (rng.standard_normal((m, k)) * rng.uniform(0.01, 30, (m, 1))).astype(np.float32)
    w = rng.standard_normal(k).astype(np.float32)
    for eps in (1e-6, 1e-5):
        y = call(gpu, x, w, eps, mem=mem)
        assert rel_l2(y, want_norm(x, w, eps)) <= 1e-6


def test_rms_norm_types_strides_and_in_place(gpu):
    rng = np.random.default_rng(2)
    m, k = 6, 2048
    x = synth.random_activation(m, k, seed=3, bf16=True)
    w = rng.standard_normal(k).astype(np.float32)
    want = want_norm(x, w, 1e-6)
    assert rel_l2(call(gpu, x, w, 1e-6, x_dtype=capi.ACT_BF16), want) <= 1e-6                       # bf16 in, f32 out
    assert rel_l2(call(gpu, x, w, 1e-6, x_dtype=capi.ACT_BF16, y_dtype=capi.ACT_BF16), want) <= 3e-3   # rounded once to bf16
    xh = x.astype(np.float16).astype(np.float32)
    assert rel_l2(call(gpu, xh, w, 1e-6, x_dtype=capi.ACT_F16, y_dtype=capi.ACT_F16), want_norm(xh, w, 1e-6)) <= 5e-4
    assert rel_l2(call(gpu, x, w, 1e-6, ldx=k + 24, ldy=k + 8, mem=capi.MEM_DEVICE), want) <= 1e-6    # row strides
    # in place on the device: y = x
    xd, wd = gpu.dev_buffer(x), gpu.dev_buffer(w)
    capi.check(gpu.L.turq_rms_norm(gpu.ctx, xd, capi.ACT_F32, m, k, k, wd, 1e-6, xd, capi.ACT_F32, k, capi.MEM_DEVICE), gpu.ctx)
    assert rel_l2(gpu.read_back(xd, (m, k), np.float32), want) <= 1e-6
    gpu.dev_free(xd)
    gpu.dev_free(wd)
    # rows of zeros stay zeros (eps keeps the root positive), huge rows stay finite
    z = np.zeros((2, k), np.float32)
    assert np.array_equal(call(gpu, z, w, 1e-6), z)
    big = (rng.standard_normal((2, k)) * 1e15).astype(np.float32)
    assert rel_l2(call(gpu, big, w, 1e-6), want_norm(big, w, 1e-6)) <= 1e-6


@pytest.mark.parametrize("k", [8, 2040, 2049, 4104, 6144, 6152, 14337])
@pytest.mark.parametrize("pad", [0, 3])
def test_rms_norm_pieces_of_a_row(gpu, k, pad):
    # a thread holds pieces of 8 columns: rows that end inside a piece or just past a round of 256 pieces (2048 columns), rows of more
    # pieces than the registers hold (above 6144), rows that 16-byte loads may not touch (an odd stride); magnitudes at which the
    # quotient by the reciprocal gives way to the plain division (rms outside 2^-60 .. 2^60)
    rng = np.random.default_rng(k + pad)
    x = rng.standard_normal((3, k)).astype(np.float32)
    w = rng.standard_normal(k).astype(np.float32)
    for scale, eps in ((1.0, 1e-6), (1e-20, 0.0)) + (((2e18, 1e-6),) if k == 8 else ()):
        xs = (x * np.float32(scale)).astype(np.float32)
        # (8 squares of up to (3 * 2e18)^2 stay below 3.4e38; squares of 1e-40 and below are f32 subnormals, 2^-149 each against 1e-40: 1e-5; else a few f32 ulps)
        bar = 1e-6 if scale >= 1.0 else 4e-5
        assert rel_l2(call(gpu, xs, w, eps, ldx=k + pad, ldy=k + pad, mem=capi.MEM_DEVICE), want_norm(xs, w, eps)) <= bar, scale


@pytest.mark.parametrize("xt,yt", [(capi.ACT_F32, capi.ACT_F32), (capi.ACT_BF16, capi.ACT_BF16), (capi.ACT_F16, capi.ACT_F16), (capi.ACT_BF16, capi.ACT_F32)])
@pytest.mark.parametrize("k", [2040, 2049, 6152])
def test_rms_norm_pieces_of_every_type(gpu, k, xt, yt):
    # rows that end inside a piece, with strides that 16-byte accesses may use (whole pieces so, the last one by element) and not
    rng = np.random.default_rng(k)
    x = synth.random_activation(5, k, seed=k, bf16=True).astype(np.float16).astype(np.float32)  # (bf16 values that f16 holds too)
    x = synth.from_bf16_bits(synth.to_bf16_bits(x)).reshape(5, k)
    w = rng.standard_normal(k).astype(np.float32)
    bar = {capi.ACT_F32: 1e-6, capi.ACT_BF16: 2.0 ** -9 + 1e-6, capi.ACT_F16: 2.0 ** -11 + 1e-6}[yt]  # one rounding of the output
    for ld in ((k + 7) // 8 * 8, k + 3):
        assert rel_l2(call(gpu, x, w, 1e-6, x_dtype=xt, y_dtype=yt, ldx=ld, ldy=ld, mem=capi.MEM_DEVICE), want_norm(x, w, 1e-6)) <= bar, ld


@pytest.mark.parametrize("xt", [capi.ACT_F32, capi.ACT_BF16, capi.ACT_F16])
@pytest.mark.parametrize("k", [520, 2048, 2304, 6144, 12288, 14336])
def test_weights_at_any_address_give_the_same_bits(gpu, k, xt):
    # a row and its weight are requested together where both allow 16-byte loads; a weight at another address is loaded by element, when it is
    # needed: to rows, and (33 rows and more, whole super-blocks) to the fragments of the prefill GEMM, one row past the last 32
    m, n = 33, 32
    x = synth.random_activation(m, k, seed=k, bf16=True)
    send = synth.to_bf16_bits(x).reshape(m, k) if xt == capi.ACT_BF16 else x.astype(np.float16) if xt == capi.ACT_F16 else x
    w = np.random.default_rng(k).standard_normal(k).astype(np.float32)
    xd, at = gpu.dev_buffer(send), [gpu.dev_buffer(w), gpu.dev_buffer(np.concatenate([np.zeros(1, np.float32), w]))]
    weights = [ctypes.c_void_p(at[0].value), ctypes.c_void_p(at[1].value + 4)]
    yd = [gpu.dev_buffer(np.zeros((m, k), np.float32)) for _ in weights]
    for wd, y in zip(weights, yd):
        capi.check(gpu.L.turq_rms_norm(gpu.ctx, xd, xt, m, k, k, wd, 1e-6, y, capi.ACT_F32, k, capi.MEM_DEVICE), gpu.ctx)
    rows = [gpu.read_back(y, (m, k), np.float32) for y in yd]
    assert np.array_equal(rows[0].view(np.uint32), rows[1].view(np.uint32))
    assert rel_l2(rows[0], want_norm(x if xt != capi.ACT_F16 else send.astype(np.float32), w, 1e-6)) <= 1e-6
    if k % 256 == 0:
        q = gpu.upload(capi.Q4_K, n, k, synth.random_weight(capi.Q4_K, n, k, seed=1), capi.LAYOUT_TILED)
        out = []
        for wd, y in zip(weights, yd):
            capi.check(gpu.L.turq_norm_qmatmul_multi(gpu.ctx, 1, (ctypes.c_void_p * 1)(q.value), xd, xt, m, k, wd, 1e-6, (ctypes.c_void_p * 1)(y.value),
                                                     capi.ACT_F32, (ctypes.c_int64 * 1)(n), None, capi.MEM_DEVICE), gpu.ctx)
            out.append(gpu.read_back(y, (m, n), np.float32))
        assert np.array_equal(out[0].view(np.uint32), out[1].view(np.uint32))
        gpu.release(q)
    for p in (xd, *at, *yd):
        gpu.dev_free(p)


def test_rms_norm_small_elements_and_signed_zeros(gpu):
    # the squares of all but four elements vanish in the sum, which makes the root exactly 3: every other element is v / 3 to the last
    # bit, whatever its size (quotients and remainders below the f32 range among them), and a zero keeps its sign
    rng = np.random.default_rng(9)
    k = 4096
    v = (rng.uniform(1, 2, k) * 2.0 ** rng.integers(-149, -29, k) * rng.choice([-1.0, 1.0], k)).astype(np.float32)
    v[4:200:2], v[5:200:2] = -0.0, 0.0
    v[200:] = np.where(np.arange(200, k) % 16 == 0, np.copysign(np.float32(0), v[200:]), v[200:])
    v[:4] = 96.0  # mean of the squares: 4 * 96^2 / 4096 = 9
    for scale in (1.0, 2.0 ** -45):  # ... and a root at which every element takes the plain division
        x = (v * np.float32(scale)).astype(np.float32).reshape(1, k)
        want = x / (np.float32(3) * np.float32(scale))
        y = call(gpu, x, np.ones(k, np.float32), 0.0, mem=capi.MEM_DEVICE)
        assert np.array_equal(y.view(np.uint32), want.view(np.uint32)), scale


@pytest.mark.parametrize("k,ldy", [(2048, 2048), (2049, 2049)])   # rows stored eight columns at a time, and element by element
def test_rms_norm_counts_every_element_that_is_no_finite_number(gpu, k, ldy):
    w = np.ones(k, np.float32)
    w[16:24], w[40:43], w[k - 1] = 1e6, 1e6, 1e6   # a whole piece of eight columns, three of another, the last column
    x = np.full((5, k), 2.0, np.float32)
    n = ctypes.c_uint64()
    capi.check(gpu.L.turq_ctx_nonfinite_count(gpu.ctx, ctypes.byref(n), 1), gpu.ctx)
    call(gpu, x, w, 1e-6, y_dtype=capi.ACT_F16, mem=capi.MEM_DEVICE, ldy=ldy)
    capi.check(gpu.L.turq_ctx_nonfinite_count(gpu.ctx, ctypes.byref(n), 1), gpu.ctx)
    assert n.value == 5 * 12


def test_rms_norm_errors(gpu):
    L, ctx = gpu.L, gpu.ctx
    x = np.zeros((2, 8), np.float32)
    w = np.ones(8, np.float32)
    y = np.zeros((2, 8), np.float32)
    args = lambda **kw: dict(dict(x=capi.ptr(x), xt=capi.ACT_F32, m=2, k=8, ldx=8, w=capi.ptr(w), eps=1e-6, y=capi.ptr(y), yt=capi.ACT_F32, ldy=8,
                                  mem=capi.MEM_HOST), **kw)
    def run(**kw):
        a = args(**kw)
        return L.turq_rms_norm(ctx, a["x"], a["xt"], a["m"], a["k"], a["ldx"], a["w"], a["eps"], a["y"], a["yt"], a["ldy"], a["mem"])
    assert run() == capi.OK
    assert run(ldx=7) == capi.ERR_SHAPE and run(ldy=7) == capi.ERR_SHAPE and run(m=-1) == capi.ERR_SHAPE
    assert run(xt=9) == capi.ERR_DTYPE and run(yt=9) == capi.ERR_DTYPE
    assert run(w=None) == capi.ERR_INVALID and run(mem=5) == capi.ERR_INVALID
    assert run(m=0) == capi.OK and run(k=0, ldx=0, ldy=0) == capi.OK
    assert L.turq_rms_norm(None, None, 0, 0, 0, 0, None, 0.0, None, 0, 0, 0) == capi.ERR_INVALID


def test_normx_from_a_gguf_file_feeds_the_projections(tmp_path):
    # the reference's order in a decoder layer: h = norm(x); q = q_proj(h)  (src/models/qwen3.rs)
    k, n = 512, 96
    rng = np.random.default_rng(9)
    nw = rng.standard_normal(k).astype("<f4")
    raw = synth.random_weight(capi.Q4_K, n, k, seed=4)
    path = tmp_path / "n.gguf"
    write_gguf(str(path), [("blk.0.attn_norm.weight", 0, (k,), nw.view(np.uint8)), ("blk.0.attn_q.weight", capi.Q4_K, (n, k), raw)])
    dev = qlinear.Device.new_hip(0)
    try:
        vb = qlinear.QVarBuilder.from_gguf(str(path), dev).pp("blk").pp(0)
        norm = qlinear.rms_norm(k, 1e-6, vb.pp("attn_norm"))
        gemma = qlinear.rms_norm(k, 1e-6, vb.pp("attn_norm"), is_gemma=True)
        q = qlinear.linear(k, n, vb.pp("attn_q"))
        assert repr(norm) == "RmsNorm" and np.array_equal(norm.weight, nw) and np.array_equal(gemma.weight, nw + np.float32(1))
        x = rng.standard_normal((2, 3, k)).astype(np.float32)
        h = norm.forward(x)
        assert h.shape == x.shape and rel_l2(h, want_norm(x, nw, 1e-6)) <= 1e-6
        from oracle import capi as orc
        y = q.forward(h)
        assert rel_l2(y, orc.matmul_dequant(capi.Q4_K, h.reshape(-1, k), raw, n, k).reshape(y.shape)) <= 1e-3
        with pytest.raises(capi.TurqError, match="shape mismatch"):
            norm.forward(np.zeros((2, k + 1), np.float32))
    finally:
        dev.close()
