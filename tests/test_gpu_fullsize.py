"""GPU parity at the full Qwen3-8B shapes the benchmark runs (decode GEMV, m = 1 and small batches).

The oracle's dense matmul finishes these in seconds on the host cores, so the comparison is direct;
the LM head (151936 x 4096) is checked on m = 1 only to keep the CPU time bounded.
"""
import numpy as np
import pytest

from oracle import capi as orc
from tests.helpers import Gpu, rel_l2
from tur_amd import capi, synth

pytestmark = pytest.mark.gpu
Q8_0, Q4_K, Q5_K, Q6_K = 8, 12, 13, 14


@pytest.fixture(scope="module")
def gpu():
    g = Gpu()
    yield g
    g.close()


CASES = [
    ("q8_0 gate 0.6B", Q8_0, 3072, 1024, [1]),
    ("q4_k gate/up 8B", Q4_K, 12288, 4096, [1, 4, 8, 16, 32]),
    ("q4_k down 8B", Q4_K, 4096, 12288, [1, 4, 16]),
    ("q4_k q/o_proj 8B", Q4_K, 4096, 4096, [1, 8, 32]),
    ("q4_k k_proj 8B", Q4_K, 1024, 4096, [1, 8, 32]),
    ("q6_k v_proj 8B", Q6_K, 1024, 4096, [1, 8, 32]),
    ("q6_k down 8B", Q6_K, 4096, 12288, [1, 8, 32]),
]


@pytest.mark.parametrize("name,dt,n,k,ms", CASES, ids=[c[0] for c in CASES])
def test_decode_shapes(gpu, name, dt, n, k, ms):
    raw = synth.random_weight(dt, n, k, seed=n + k + dt)
    w = gpu.upload(dt, n, k, raw, capi.LAYOUT_TILED)
    for m in ms:
        x = synth.random_activation(m, k, seed=m)
        y = gpu.qmatmul(w, x, n, k)
        dense = orc.matmul_dequant(dt, x, raw, n, k)
        assert rel_l2(y, dense) <= 1e-3
        xb = synth.random_activation(m, k, seed=m + 1, bf16=True)
        yb = gpu.qmatmul(w, xb, n, k, x_dtype=capi.ACT_BF16)
        assert rel_l2(yb, orc.matmul_dequant(dt, xb, raw, n, k)) <= 2e-5
        if m == ms[0]:
            assert rel_l2(y, orc.qmatmul(dt, x, raw, n, k)) <= 1e-2
    gpu.release(w)


@pytest.mark.parametrize("dt", [Q6_K, Q5_K], ids=["q6_k", "q5_k"])
def test_lm_head(gpu, dt):
    n, k = 151936, 4096
    raw = synth.random_weight(dt, n, k, seed=dt)
    w = gpu.upload(dt, n, k, raw, capi.LAYOUT_TILED)
    x = synth.random_activation(1, k, seed=9, bf16=True)
    y = gpu.qmatmul(w, x, n, k, x_dtype=capi.ACT_BF16)
    assert rel_l2(y, orc.matmul_dequant(dt, x, raw, n, k)) <= 2e-5
    # m = 16: spot-check 4096 vocabulary rows spread over the matrix against the oracle
    x16 = synth.random_activation(16, k, seed=10, bf16=True)
    y16 = gpu.qmatmul(w, x16, n, k, x_dtype=capi.ACT_BF16)
    rows = np.arange(0, n, n // 4096)[:4096]
    sub = raw.reshape(n, -1)[rows].reshape(-1)
    assert rel_l2(y16[:, rows], orc.matmul_dequant(dt, x16, sub, len(rows), k)) <= 2e-5
    # m = 128: the prefill GEMM of this format (the wide 128 x 256 tile at this shape), same spot check on the
    # f32 result; the configuration's bf16 output is that result rounded once, bit for bit
    x128 = synth.random_activation(128, k, seed=11, bf16=True)
    y128 = gpu.qmatmul(w, x128, n, k, x_dtype=capi.ACT_BF16)
    yb128 = gpu.qmatmul(w, x128, n, k, x_dtype=capi.ACT_BF16, y_dtype=capi.ACT_BF16)
    assert np.all(np.isfinite(y128))
    assert rel_l2(y128[:, rows], orc.matmul_dequant(dt, x128, sub, len(rows), k)) <= 1e-3
    assert np.array_equal(synth.to_bf16_bits(y128).reshape(128, n), synth.to_bf16_bits(yb128).reshape(128, n))
    gpu.release(w)


@pytest.mark.parametrize("m", [512, 2048])
def test_prefill_up_proj(gpu, m):
    # Q4_K up_proj 12288 x 4096, bf16 activations [m, 4096]; the oracle checks every 16th
    # weight row (768 rows spread over all workgroups) to keep the CPU time bounded
    n, k = 12288, 4096
    raw = synth.random_weight(Q4_K, n, k, seed=44)
    w = gpu.upload(Q4_K, n, k, raw, capi.LAYOUT_TILED)
    x = synth.random_activation(m, k, seed=m, bf16=True)
    y = gpu.qmatmul(w, x, n, k, x_dtype=capi.ACT_BF16)
    # the configuration's own output type: f32 sums stored as bf16, i.e. the f32 result rounded once (to nearest even)
    yb = gpu.qmatmul(w, x, n, k, x_dtype=capi.ACT_BF16, y_dtype=capi.ACT_BF16)
    gpu.release(w)
    rows = np.arange(5, n, 16)
    sub = raw.reshape(n, -1)[rows].reshape(-1)
    want = orc.matmul_dequant(Q4_K, x, sub, len(rows), k)
    assert np.all(np.isfinite(y))
    assert rel_l2(y[:, rows], want) <= 1e-3
    assert np.array_equal(synth.to_bf16_bits(y).reshape(m, n), synth.to_bf16_bits(yb).reshape(m, n))
    assert rel_l2(yb[:, rows], synth.from_bf16_bits(synth.to_bf16_bits(want)).reshape(want.shape)) <= 1.5e-3


@pytest.mark.parametrize("m", [64, 128, 256])
def test_prefill_down_proj_split_columns(gpu, m):
    # the tall matrix of the layer (Q6_K down_proj 4096 x 12288) at prompt-chunk sizes: few workgroup tiles, so every tile's
    # columns go to the waves of its workgroup (tiles of 32 x 32, 64 x 32 and 64 x 64); the oracle checks every 16th weight row
    n, k = 4096, 12288
    raw = synth.random_weight(Q6_K, n, k, seed=45)
    w = gpu.upload(Q6_K, n, k, raw, capi.LAYOUT_TILED)
    x = synth.random_activation(m, k, seed=m, bf16=True)
    y = gpu.qmatmul(w, x, n, k, x_dtype=capi.ACT_BF16)
    y2 = gpu.qmatmul(w, x, n, k, x_dtype=capi.ACT_BF16)
    yb = gpu.qmatmul(w, x, n, k, x_dtype=capi.ACT_BF16, y_dtype=capi.ACT_BF16)
    gpu.release(w)
    rows = np.arange(3, n, 16)
    sub = raw.reshape(n, -1)[rows].reshape(-1)
    want = orc.matmul_dequant(Q6_K, x, sub, len(rows), k)
    assert np.all(np.isfinite(y))
    assert rel_l2(y[:, rows], want) <= 1e-3
    assert np.array_equal(y, y2)
    assert np.array_equal(synth.to_bf16_bits(y).reshape(m, n), synth.to_bf16_bits(yb).reshape(m, n))


# one Qwen3-8B decoder layer of a Q4_K_M file
LAYER = [("q", Q4_K, 4096, 4096), ("k", Q4_K, 1024, 4096), ("v", Q6_K, 1024, 4096), ("o", Q4_K, 4096, 4096),
         ("gate", Q4_K, 12288, 4096), ("up", Q4_K, 12288, 4096), ("down", Q6_K, 4096, 12288)]


@pytest.fixture(scope="module")
def layer(gpu):
    raws = {lb: synth.random_weight(dt, n, k, seed=300 + i) for i, (lb, dt, n, k) in enumerate(LAYER)}
    ws = {lb: gpu.upload(dt, n, k, raws[lb], capi.LAYOUT_TILED) for lb, dt, n, k in LAYER}
    yield raws, ws
    for w in ws.values():
        gpu.release(w)


@pytest.mark.parametrize("x_dtype", [capi.ACT_F32, capi.ACT_BF16], ids=["f32", "bf16"])
@pytest.mark.parametrize("m", [1, 4, 8, 16, 32, 40, 64, 128, 256])
def test_q4km_decoder_layer_grouped_calls(gpu, layer, m, x_dtype):
    # the layer's seven linears driven as the reference's decoder layer drives them (src/models/qwen3.rs:272-274, 161-167):
    # q / k / v on one tensor through turq_qmatmul_multi (two formats in one launch), o_proj alone, gate / up through
    # turq_qmatmul_multi, down_proj alone; device pointers, every output against the f32 matmul on the dequantized weights
    raws, ws = layer
    # (40 and 64 rows: gate / up in two chunks through the kernels of up to 32 rows, the others through the prefill GEMM, whose
    # folded f16 scales cost about 3e-4; down_proj, o_proj and q / k / v with their columns split over the waves;
    # 128 and 256 rows: gate and up as one GEMM launch over the rows of both)
    bf = x_dtype == capi.ACT_BF16
    bar = 2e-5 if bf and m <= 32 else 1e-3
    shape = {lb: (dt, n, k) for lb, dt, n, k in LAYER}
    for gi, group in enumerate((("q", "k", "v"), ("o",), ("gate", "up"), ("down",))):
        k = shape[group[0]][2]
        x = synth.random_activation(m, k, seed=17 * m + gi, bf16=bf)
        ns = [shape[lb][1] for lb in group]
        if len(group) > 1:
            outs = gpu.qmatmul_multi([ws[lb] for lb in group], x, ns, k, x_dtype=x_dtype)
        else:
            outs = [gpu.qmatmul_device(ws[group[0]], x, ns[0], k, x_dtype=x_dtype)]
        for lb, y in zip(group, outs):
            dt, n, _ = shape[lb]
            assert y.shape == (m, n)
            assert rel_l2(y, orc.matmul_dequant(dt, x, raws[lb], n, k)) <= (2e-5 if bf and m <= 64 and lb in ("gate", "up") else bar), (lb, m)


@pytest.mark.parametrize("m", [128, 1024])
def test_prefill_gate_and_up_in_one_launch(gpu, layer, m):
    # gate and up of a prompt chunk through turq_qmatmul_multi are ONE launch of the prefill GEMM over the rows of both where that
    # fills the machine better (128 rows: each alone leaves CUs idle; 1024 rows: the wide tile then fills its rounds exactly);
    # against the single calls - other tiles, so another order of the f32 sums where the waves of a workgroup split k - and
    # against the oracle on every 16th weight row
    raws, ws = layer
    n, k = 12288, 4096
    x = synth.random_activation(m, k, seed=900 + m, bf16=True)
    yg, yu = gpu.qmatmul_multi([ws["gate"], ws["up"]], x, [n, n], k, x_dtype=capi.ACT_BF16)
    rows = np.arange(7, n, 16)
    for lb, y in (("gate", yg), ("up", yu)):
        single = gpu.qmatmul_device(ws[lb], x, n, k, x_dtype=capi.ACT_BF16)
        assert rel_l2(y, single) <= 2e-6, (lb, rel_l2(y, single))
        sub = raws[lb].reshape(n, -1)[rows].reshape(-1)
        assert rel_l2(y[:, rows], orc.matmul_dequant(Q4_K, x, sub, len(rows), k)) <= 1e-3, lb


def test_mlp_gate_up_and_token_embd(gpu):
    # the two calls that widen the path, at Qwen3-8B sizes: gate / up with SiLU (12288 x 4096 Q4_K: one launch at every row count
    # here - the one-row kernel, the staged rows kernel with six tiles per workgroup, its four-wave form from 17 rows on) and
    # token_embd rows (151936 x 4096 Q6_K) against the full dequantize
    from oracle import oracle_np as onp
    n, k = 12288, 4096
    raw_g = synth.random_weight(Q4_K, n, k, seed=1)
    raw_u = synth.random_weight(Q4_K, n, k, seed=2)
    wg = gpu.upload(Q4_K, n, k, raw_g, capi.LAYOUT_TILED)
    wu = gpu.upload(Q4_K, n, k, raw_u, capi.LAYOUT_TILED)
    for m in (1, 2, 5, 16, 17, 32, 33, 64):      # (33, 64: two chunks of up to 32 rows)
        x = synth.random_activation(m, k, seed=40 + m, bf16=True)
        y = gpu.gate_up(wg, wu, x, n, k, x_dtype=capi.ACT_BF16)
        want = onp.silu_mul(orc.matmul_dequant(Q4_K, x, raw_g, n, k), orc.matmul_dequant(Q4_K, x, raw_u, n, k))
        assert rel_l2(y, want) <= 5e-5, m
    gpu.release(wg)
    gpu.release(wu)
    n = 151936
    raw = synth.random_weight(Q6_K, n, k, seed=3)
    w = gpu.upload(Q6_K, n, k, raw, capi.LAYOUT_NATIVE)
    ids = np.concatenate([[0, n - 1], np.random.default_rng(4).integers(0, n, 510)]).astype(np.uint32)
    out = np.zeros((len(ids), k), np.float32)
    capi.check(gpu.L.turq_embedding_lookup(gpu.ctx, w, capi.ptr(ids), len(ids), capi.ptr(out), capi.ACT_F32, k, capi.MEM_HOST), gpu.ctx)
    rows = raw.reshape(n, -1)[ids].reshape(-1)
    assert np.array_equal(out.view(np.uint32), orc.dequantize(Q6_K, rows).reshape(len(ids), k).view(np.uint32))
    gpu.release(w)
