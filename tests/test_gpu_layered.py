"""The LAYERED contraction (kernels_layered.hip) against the CPU oracle where
it can go wrong: input widths that end inside a contraction step (with
infinities, which the zero rows past the input must not meet), output widths
that end inside a tile, rows at every alignment (16-byte pieces, 4-byte
pieces, elements), the small and the large workgroup tile, epilogues on the
accumulators and in the loop over the finished tile, a bias that seeds the
sum.  Bars: those of test_gpu_parity.py (fp64 1e-12 relative to the largest
value)."""
import numpy as np
import pytest

import oracle
import ponni_amd as P
from ponni_amd import graph as G
from tests.test_gpu_parity import ORACLE_MODE, TORCH_DT, check_f32, check_half, check_non_finite, gpu_run
from tests.test_graph import lowered_with_params

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _oracle_built():
    oracle.build()


def _w(r, a, b):
    return r.uniform(-1, 1, (a, b)) * np.sqrt(6.0 / (a + b))


def _generated(r, n_in, w):
    g = G.GraphBuilder(n_in)
    h = g.unary("Tanh", g.dense(g.input, _w(r, w, n_in), r.uniform(-0.2, 0.2, w), name="a"))
    return lowered_with_params(g.finish(g.unary("Abs", g.dense(h, _w(r, 5, w), r.uniform(-0.2, 0.2, 5), name="b"))))


CHAINS = {
    # usual steps, then steps of the loop (two with parameters), then usual ones in the loop
    "epilogues": lambda r: [P.Matvec(_w(r, 37, 150)), P.Bias(r.uniform(-0.1, 0.1, 150)), P.Silu(150), P.Mish(150),
                            P.Bias(r.uniform(-0.1, 0.1, 150)), P.Tanh(150), P.Matvec(_w(r, 150, 70)), P.Gelu(70),
                            P.Matvec(_w(r, 70, 3)), P.Bias(r.uniform(-0.1, 0.1, 3)), P.LeakyRelu(3, 0.2)],
    "one_step": lambda r: [P.Matvec(_w(r, 3, 65)), P.Sigmoid(65), P.LayerNorm(65), P.Matvec(_w(r, 65, 129))],
    "generated": lambda r: _generated(r, 50, 200),
    "projection": lambda r: [P.Save_State(0, 9), P.Matvec(_w(r, 9, 33)), P.Relu(33),
                             P.Binop_Projection_Add(0, _w(r, 9, 33), r.uniform(-0.1, 0.1, 33)),
                             P.Matvec(_w(r, 33, 17)), P.Gelu(17, True)],
}


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16", "f64"])
@pytest.mark.parametrize("chain", sorted(CHAINS))
def test_layered_edges(cuda, chain, dtype):
    layers = CHAINS[chain](np.random.default_rng(31))
    # the last batch has enough columns for the large tile (512 of them)
    for B, pad in [(1, 0), (127, 0), (130, 6), (257, 3), (33_003, 5), (40_000, 0)]:
        x = np.random.default_rng(B).standard_normal((layers[0].n_in, B))
        print(f"layered: chain={chain} dtype={dtype} B={B}", flush=True)
        got, xg, m = gpu_run(layers, x, dtype=dtype, path="layered", pad=pad)
        assert m.path == "layered"
        want = oracle.forward(layers, xg, ORACLE_MODE[dtype])
        if dtype == "f32":
            check_f32(got, want)
        elif dtype == "f64":
            assert np.abs(got - want).max() <= 1e-12 * max(1.0, np.abs(want).max())
        else:
            check_half(got, want)


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16", "f64"])
@pytest.mark.parametrize("n_in", [5, 16, 33])
def test_layered_infinite_inputs(cuda, n_in, dtype):
    r = np.random.default_rng(n_in)
    layers = [P.Matvec(_w(r, n_in, 70)), P.Tanh(70), P.Matvec(_w(r, 70, 21)), P.Bias(r.uniform(-0.1, 0.1, 21))]
    x = r.standard_normal((n_in, 515))
    x[r.integers(n_in, size=200), np.arange(0, 400, 2)] = np.where(np.arange(200) % 2, np.inf, -np.inf)
    print(f"layered infinities: n_in={n_in} dtype={dtype}", flush=True)
    for pad in (0, 5):
        got, xg, _ = gpu_run(layers, x, dtype=dtype, path="layered", pad=pad)
        want = oracle.forward(layers, xg, ORACLE_MODE[dtype])
        assert np.isfinite(want[:, 0:400:2]).mean() > 0.5
        check_non_finite(got, want, dtype)


@pytest.mark.parametrize("dtype", ["f32", "f16", "f64"])
@pytest.mark.parametrize("n_out", [64, 65, 128])
def test_layered_one_layer_in_place(cuda, n_out, dtype):
    """A chain of one layer whose outputs take its inputs' rows: the outputs of a
    column, read by every workgroup that computes one of them, stay in one."""
    import torch

    r = np.random.default_rng(n_out)
    m = P.create_inference_model(P.Matvec(_w(r, 200, n_out)), P.Relu(n_out), dtype=dtype, path="layered")
    for B in (130, 2_000):
        print(f"layered in place: n_out={n_out} dtype={dtype} B={B}", flush=True)
        x = torch.randn((200, B), device="cuda:0", generator=torch.Generator("cuda:0").manual_seed(B))
        x = x.to(getattr(torch, TORCH_DT[dtype]))
        want = m.forward_batch_parallel(x)
        m.forward_batch_parallel(x, x[:n_out])
        torch.cuda.synchronize()
        assert torch.equal(x[:n_out], want)


# (largest relative error in fp32 ulps of 2^-24: 1 + e and the quotient round to
# 1, 2^x is off by 1 or 2 and, carried along, its argument by a half, and tanh's last
# addition rounds to a half of at least 0.5; the hardware forms alone: 5.8, 31, 63)
FP32_BOUNDS = [("tanh", 1e-6, 0.55, 2), ("tanh", -2.0, -0.55, 4.5), ("tanh", -8.0, -2.0, 2), ("sigmoid", -40.0, -6.0, 5),
               ("silu", -80.0, -40.0, 6), ("sigmoid", -3.0, 9.0, 5), ("silu", -6.0, 9.0, 6), ("gelu", -0.5, 6.0, 6)]


def _activation_error(cuda, dtype, act, lo, hi):
    """y, the exact value and x of one activation on both signs or as given,
    through an identity layer (exact in any order of its sum)."""
    import torch

    n = 64
    layer = {"tanh": P.Tanh(n), "sigmoid": P.Sigmoid(n), "silu": P.Silu(n), "gelu": P.Gelu(n, True)}[act]
    m = P.create_inference_model(P.Matvec(np.eye(n)), layer, dtype=dtype, path="layered")
    gen = torch.Generator("cuda:0").manual_seed(5)
    x = torch.rand((n, 20_000), device="cuda:0", dtype=torch.float64, generator=gen) * (hi - lo) + lo
    x = x.to(getattr(torch, TORCH_DT[dtype]))
    y = m.forward_batch_parallel(x).double()
    v = x.double()
    u = 2 * np.sqrt(2 / np.pi) * (v + 0.044715 * v**3)
    want = {"tanh": torch.tanh, "sigmoid": lambda v: 1 / (1 + torch.exp(-v)), "silu": lambda v: v / (1 + torch.exp(-v)),
            "gelu": lambda v: v / (1 + torch.exp(-u))}[act](v)
    return y, want


@pytest.mark.parametrize("act, lo, hi, ulps", FP32_BOUNDS)
def test_layered_fp32_activations(cuda, act, lo, hi, ulps):
    y, want = _activation_error(cuda, "f32", act, lo, hi)
    assert float(((y - want).abs() / want.abs()).max()) * 2**24 <= ulps


@pytest.mark.parametrize("dtype, digits, smallest", [("f16", 10, -14), ("bf16", 7, -126)])
@pytest.mark.parametrize("lo, hi", [(1e-7, 1e-5), (1e-5, 1e-4), (1e-4, 1e-3), (1e-3, 0.1), (-2.0, 2.0)])
def test_layered_half_tanh_near_zero(cuda, lo, hi, dtype, digits, smallest):
    """Half an ulp of the type, and a sixteenth for fp32's own error (x for
    tanh(x) below 2^-7: a third of x^2, 1/25 of an fp16 ulp; above, an fp32 ulp of
    one: 1/30 of one).  The hardware form alone was off by 2 ulps at 1e-4."""
    import torch

    y, want = _activation_error(cuda, dtype, "tanh", lo, hi)
    ulp = torch.exp2(torch.floor(torch.log2(want.abs())).clamp_min(smallest) - digits)
    assert float(((y - want).abs() / ulp).max()) <= 0.5 + 1 / 16
