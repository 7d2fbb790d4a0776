"""The grouped GEMM's two tile kernels at the sizes where they can go wrong:
expert loads at the edges of the small-tile GEMM's operands (8 pairs packed hi
and lo in one operand, 16 pairs per tile) and just past them, empty experts, a
K that ends inside an A chunk, merged shared tiles; and the same loads doubled,
past the rule that selects the small tiles (11 to 12 pairs per expert). Against the
oracle, to the repository's bar, and every row closely; the dispatch's choice between
the two kernels on both sides of its tile counts; and GGUF-order weights (a cached layer) bit for
bit against the tiled copies (a resident one)."""
import numpy as np
import pytest

from ingot_amd import configs as CF
from ingot_amd.moe import (IQ2_S, IQ2_XS, IQ3_S, IQ3_XXS, IQ4_NL, IQ4_XS, Q4_K, Q5_K, Q6_K, Q8_0, STAGE_DOWN, STAGE_GATEUP,
                           MoeLayer)
from util import check_layer

pytestmark = pytest.mark.gpu

LOADS = [1, 7, 8, 9, 15, 16, 17, 31, 32, 33, 0, 5, 0, 0, 1, 2]  # 177 pairs, 11.1 per expert


def routed_inputs(spec, loads, H, seed):
    """Inputs whose identity router sends loads[e] tokens to expert e (top-1)."""
    E = len(loads)
    T = sum(loads)
    spec.router = np.zeros((E, H), np.float32)
    spec.router[np.arange(E), np.arange(E)] = 1.0
    x = CF.inputs(seed, T, H) * 0.05
    order = np.repeat(np.arange(E), loads)
    np.random.default_rng(seed).shuffle(order)
    x[:, :E] = 0.0
    x[np.arange(T), order] = 4.0
    return x


def assert_rows_close(spec, x, out, oracle):
    """Every row within 2^-15 of 64 bits. The split operands' products and the 32-bit
    sums are good to about 2^-21 of the terms' size, and a row's terms cancel: the q and
    min products of Q4_K and Q5_K (weights of +-2.5 sigma around a block's minimum) to
    about 2^-2, a row whose g or u is small for its x to some 2^-4 of its terms in these
    few hundred rows. A row whose lo parts were lost would be off by 2^-11 / sqrt(12), 2^-13."""
    st, ref, _, _ = oracle.moe_forward(spec, x, oracle.F64)
    assert st == 0
    err = np.linalg.norm(out - ref, axis=1) / np.linalg.norm(ref, axis=1)
    assert err.max() <= 2.0 ** -15, f"row {err.argmax()}: {err.max():.2e}"


@pytest.mark.parametrize("gk,dk,F", [(Q4_K, Q4_K, 256), (Q5_K, Q5_K, 768), (Q6_K, Q6_K, 256), (Q4_K, Q6_K, 768),
                                     (IQ2_XS, IQ2_XS, 512), (IQ2_S, IQ2_S, 512), (IQ3_XXS, IQ4_NL, 192),
                                     (IQ3_S, IQ3_S, 512), (IQ4_XS, IQ4_XS, 256), (IQ4_NL, IQ4_NL, 64)])
@pytest.mark.parametrize("shared", [False, True])
def test_tile_loads(gpu, oracle, gk, dk, F, shared):
    base = LOADS + [0] * (16 if gk == Q6_K else 0)  # Q6_K gate/up: up to 6 pairs per expert
    H, E = 1024, len(base)
    spec = CF.make_layer(61, 0, H, E, 1, F, gk, dk, shared_ffn=F if shared else 0)
    for times in (1, 2):  # small tiles; past the rule
        loads = [times * v for v in base]
        x = routed_inputs(spec, loads, H, 61 + times)
        res, cached = MoeLayer(gpu, spec), MoeLayer(gpu, spec, cache_slots=5)
        out, ids, _ = check_layer(res, spec, x, oracle, f"{gk}/{dk} F={F} shared={shared} {times}x loads")
        assert np.array_equal(np.bincount(ids.ravel(), minlength=E), loads)
        assert_rows_close(spec, x, out, oracle)
        gemm = "k_gemm_small" if times == 1 else "k_gemm_f16"
        assert res.stage_kernel(STAGE_GATEUP) == f"{gemm}<gate_up>" and res.stage_kernel(STAGE_DOWN) == f"{gemm}<down>"
        assert np.array_equal(out, cached(x)[0]), "GGUF order against tiled copies"
        res.destroy()
        cached.destroy()


def wide_spec(gk, dk, shared):
    """64 experts of 1792, four of them distinct."""
    spec = CF.make_layer(66, 0, 1024, 4, 1, 1792, gk, dk, shared_ffn=1792 if shared else 0)
    spec.experts = 64
    for m in ("gate", "up", "down"):
        setattr(spec, m, getattr(spec, m).select([(5 * e) % 4 for e in range(64)]))
    return spec


# 64 experts of 1792 (28 gate/up blocks a tile): the dispatch chooses from 686 pairs on, k_gemm_f16 above
# 54 tiles of 16 pairs if they are more than 7 to 4 64-pair tiles.
@pytest.mark.parametrize("loads,shared,f16", [
    ([12] * 64, False, False),
    ([224, 224, 240] + [1] * 11, False, False), ([224, 224, 240] + [1] * 12, False, True),  # 54 tiles; 55
    ([48] * 12 + [6] * 20, False, False), ([48] * 13 + [4] * 18, False, True),  # 56 to 32; 57 to 31
    ([250, 250, 240] + [1] * 27, True, True)])
@pytest.mark.parametrize("gk,dk", [(Q4_K, Q6_K), (Q8_0, Q8_0)])
def test_dispatch_chooses_by_tiles(gpu, oracle, gk, dk, loads, shared, f16):
    spec = wide_spec(gk, dk, shared)
    H, E = spec.hidden, spec.experts
    loads = loads + [0] * (E - len(loads))
    x = routed_inputs(spec, loads, H, 66)
    res, cached = MoeLayer(gpu, spec), MoeLayer(gpu, spec, cache_slots=40)
    out, ids, _ = res(x)
    assert np.array_equal(np.bincount(ids.ravel(), minlength=E), loads)
    gemm = "k_gemm_f16" if f16 else "k_gemm_small"
    assert res.stage_kernel(STAGE_GATEUP) == f"{gemm}<gate_up>" and res.stage_kernel(STAGE_DOWN) == f"{gemm}<down>"
    assert_rows_close(spec, x, out, oracle)
    assert np.array_equal(out, cached(x)[0])
    res.destroy()
    cached.destroy()


def test_captured_forward_chooses_at_each_replay(gpu):
    """One graph, replayed with inputs for which the dispatch chooses either kernel."""
    spec = wide_spec(Q4_K, Q6_K, True)
    T, H, E = 768, spec.hidden, spec.experts
    xs = [routed_inputs(spec, loads + [0] * (E - len(loads)), H, 67)
          for loads in ([12] * 64, [250, 250, 241] + [1] * 27, [256, 256, 256])]
    eager, layer = MoeLayer(gpu, spec), MoeLayer(gpu, spec)
    refs = [eager(x)[0] for x in xs]
    layer.reserve(T)
    dx, dout = gpu.buffer(4 * T * H), gpu.buffer(4 * T * H)
    gpu.graph_begin()
    layer.forward(dx, T, dout)
    graph = gpu.graph_end()
    for i in (0, 1, 0, 2, 1):
        dx.upload(xs[i])
        graph.launch()
        gpu.synchronize()
        assert np.array_equal(dout.download(np.float32, T * H).reshape(T, H), refs[i])
        gemm = ("k_gemm_small", "k_gemm_f16", "k_gemm_f16")[i]  # 112 tiles to 76; 123 to 51; 96 to 24
        assert layer.stage_kernel(STAGE_GATEUP) == f"{gemm}<gate_up>"
        assert np.array_equal(eager(xs[i])[0], refs[i])
    gpu.check_device_flags()
    graph.destroy()
    eager.destroy()
    layer.destroy()
