"""Q8_0 on the f16 GEMM (exact int8 operands, act split by each row's own
maximum): routed experts on small and 64-pair tiles, resident and cached, merged
shared expert; a gated Q8_0 shared expert beside routed experts of other formats,
whose x is stored in that format's column order; and activations of any scale,
which raise no range flag."""
import numpy as np
import pytest

from ingot_amd import configs as CF
from ingot_amd.moe import IQ2_XS, IQ4_NL, Q4_K, Q6_K, Q8_0, STAGE_DOWN, STAGE_GATEUP, Gpu, LayerSpec, Matrix, MoeLayer
from test_gpu_small_tiles import LOADS, assert_rows_close, routed_inputs
from util import check_layer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("F,shared", [(64, 0), (192, 192), (768, 256)])
def test_q8_routed(gpu, oracle, F, shared):
    H, E = 1024, len(LOADS)
    spec = CF.make_layer(62, 0, H, E, 1, F, Q8_0, Q8_0, shared_ffn=shared)
    blocks = spec.gate.data.reshape(-1, 34)
    blocks[::7, :2] = 0  # zero scales
    blocks[1::9, 2:] = 0x80  # every value -128
    for times in (1, 2):  # 16-pair tiles; 64-pair tiles
        x = routed_inputs(spec, [times * v for v in LOADS], H, 62 + times)
        res, cached = MoeLayer(gpu, spec), MoeLayer(gpu, spec, cache_slots=5)
        out, _, _ = check_layer(res, spec, x, oracle, f"Q8_0 F={F} shared={shared} {times}x loads")
        assert_rows_close(spec, x, out, oracle)
        gemm = "k_gemm_small" if times == 1 else "k_gemm_f16"
        assert res.stage_kernel(STAGE_GATEUP) == f"{gemm}<gate_up>" and res.stage_kernel(STAGE_DOWN) == f"{gemm}<down>"
        assert np.array_equal(out, cached(x)[0])
        res.destroy()
        cached.destroy()


@pytest.mark.parametrize("gk,dk", [(IQ2_XS, IQ2_XS), (Q6_K, Q6_K), (Q4_K, Q4_K), (Q4_K, Q8_0), (IQ4_NL, IQ4_NL)])
def test_q8_shared_beside_other_formats(gpu, oracle, gk, dk):
    spec = CF.make_layer(63, gk, 2048, 32, 8, 512, gk, dk, shared_ffn=256, shared_gate_kind=Q8_0,
                         shared_down_kind=Q8_0, shared_gated=True)
    res, cached = MoeLayer(gpu, spec), MoeLayer(gpu, spec, cache_slots=5)
    for T in (9, 17, 130, 300):  # one and four 16-token tiles per block
        x = CF.inputs(63, T, 2048, seed=T)
        out, _, _ = check_layer(res, spec, x, oracle, f"Q8_0 shared beside {gk}/{dk} T={T}")
        assert np.array_equal(out, cached(x)[0])
    res.destroy()
    cached.destroy()


@pytest.mark.parametrize("H,F,SF,T", [
    (2048, 256, 64, 17), (2048, 256, 64, 200),     # one 64-column slab; down on the fp32 GEMM from 129 tokens
    (2048, 256, 192, 70), (2048, 512, 320, 250),   # superblocks cut short; four tiles a block, the last in part (down)
    (2048, 512, 320, 700),                         # four tiles a block (gate/up), down on the fp32 GEMM
    (4096, 512, 512, 100), (4096, 512, 512, 450),  # wider x; four tiles a block (down; both)
    (1024, 512, 512, 2048)])                       # the fp32 GEMM's rounds full: neither
def test_q8_shared_shapes(gpu, oracle, H, F, SF, T):
    """The shared expert's kernels at the edges of the rules that choose them."""
    K = 4 if T <= 64 else 1  # more than 64 pairs: not the decode kernels
    spec = CF.make_layer(65, 0, H, 8, K, F, Q4_K, Q4_K, shared_ffn=SF, shared_gate_kind=Q8_0, shared_down_kind=Q8_0,
                         shared_gated=True)
    x = CF.inputs(65, T, H, seed=SF)
    res, cached = MoeLayer(gpu, spec), MoeLayer(gpu, spec, cache_slots=3)
    out, _, _ = res(x)
    assert_rows_close(spec, x, out, oracle)
    assert np.array_equal(out, cached(x)[0])
    res.destroy()
    cached.destroy()


def test_q8_expert_of_4_gib(gpu):
    """Matrices whose bytes do not fit the f16 GEMM's 32-bit offsets stay on the fp32 GEMM:
    an expert with only its last 64 columns of act in use, at 4 GiB into gate and up."""
    H, F = 1024, 1 << 22
    gate, up, down = (np.zeros(n, np.uint8) for n in (F * 1088, F * 1088, H * (F // 32 * 34)))
    rng = np.random.default_rng(68)
    scale = np.frombuffer(np.float16(0.002).tobytes(), np.uint8)
    values = []
    for m, rows, blocks in ((gate, slice(F - 64, F), slice(0, 32)), (up, slice(F - 64, F), slice(0, 32)),
                            (down, slice(0, H), slice(F // 32 - 2, F // 32))):
        b = m.reshape(-1, H // 32 if m is not down else F // 32, 34)[rows, blocks]
        b[..., :2] = scale
        b[..., 2:] = rng.integers(0, 256, b.shape[:2] + (32,))
        values.append(b[..., 2:].view(np.int8).reshape(len(b), -1) * np.float64(np.float16(0.002)))
    mats = [Matrix(gate, H, F, 1, Q8_0, 1088), Matrix(up, H, F, 1, Q8_0, 1088), Matrix(down, F, H, 1, Q8_0, F // 32 * 34)]
    x = CF.inputs(68, 3, H)
    layer = MoeLayer(gpu, LayerSpec(hidden=H, experts=1, top_k=1, router=np.zeros((1, H), np.float32), gate=mats[0],
                                    up=mats[1], down=mats[2]))
    out = layer(x)[0]
    g, u = x @ values[0].T, x @ values[1].T
    ref = (g / (1.0 + np.exp(-g)) * u) @ values[2].T
    assert np.linalg.norm(out - ref) <= 1e-5 * np.linalg.norm(ref)  # two 32-bit sums of at most 1024 products
    assert layer.stage_kernel(STAGE_GATEUP) == "k_gemm<gate_up>"
    layer.destroy()


def test_q8_copies_leave_room():
    """The second copies of a Q8_0 layer's weights are not made on a nearly full card (a
    sixteenth of it is left), and the layer computes the same without them."""
    spec = CF.make_layer(67, 0, 1024, 32, 4, 512, Q8_0, Q8_0)
    x = CF.inputs(67, 70, 1024)
    gpu = Gpu(0)  # its own: a failed allocation closes a context
    full, roomy = MoeLayer(gpu, spec), MoeLayer(gpu, spec)
    bytes_ = full.weight_bytes()
    roomy.reserve(70)
    total = gpu.mem_info()[1]
    fill = []
    for _ in range(64):  # nothing touches it
        left = gpu.mem_info()[0] - total // 16 - (8 << 20)
        if left < 2 << 20:
            break
        fill.append(gpu.buffer(min(left, 32 << 30)))
    out = full(x)[0]
    kept, avail = full.weight_bytes(), gpu.mem_info()[0]
    clone = roomy.clone()  # its weights, without their copies
    cloned = clone.weight_bytes()
    for b in fill:
        b.free()
    assert kept == bytes_ and avail > total // 16 - (16 << 20)  # less the workspace
    assert cloned == bytes_ and np.array_equal(out, clone(x)[0])
    assert np.array_equal(out, roomy(x)[0]) and roomy.weight_bytes() > 2 * bytes_ - (1 << 20)
    for layer in (full, roomy, clone):
        layer.destroy()
    gpu.close()


@pytest.mark.parametrize("scale", [1e-12, 1e-4, 1e4, 1e12])
def test_q8_any_activation_scale(gpu, oracle, scale):
    """No token-wise guess of the activations' size enters: the relative error
    stays that of the usual scale (two 32-bit sums of at most 1024 products)."""
    spec = CF.make_layer(64, 0, 1024, 16, 4, 256, Q8_0, Q8_0)
    x = (CF.inputs(64, 40, 1024) * np.float32(scale)).astype(np.float32)
    layer = MoeLayer(gpu, spec)
    out, ids, _ = layer(x)
    assert not layer.last_fallback
    st, ref, rids, _ = oracle.moe_forward(spec, x, oracle.F64)
    assert st == 0 and np.array_equal(ids, rids)
    assert np.linalg.norm(out - ref) <= 1e-5 * np.linalg.norm(ref)
    layer.destroy()
