"""The small-batch kernels of FUSED plans (fused_split.h: a workgroup's waves
share one tile of columns) against the CPU oracle, and the kernels that large
batches run on the same small batches: tile counts that do and do not divide
among the waves, padded widths, projections, barriers, saved states, a
transposed output, one and two column tiles, ragged column edges.

A plan put on the device by ponni_plan_device_params has only its main
kernel loaded, and the allocation-free forward loads nothing, so that pair
runs the main kernel at any batch; ponni_forward chooses by the batch.
Bars: those of test_gpu_parity.py (fp64 1e-12 relative to the largest value)."""
import ctypes

import numpy as np
import pytest

import oracle
import ponni_amd as P
from tests.test_gpu_parity import ORACLE_MODE, TORCH_DT, check_f32, check_half

pytestmark = pytest.mark.gpu


def _w(r, a, b):
    return r.uniform(-1, 1, (a, b)) * np.sqrt(6.0 / (a + b))


def _mlp(r, widths, act):
    layers = []
    for i, (a, b) in enumerate(zip(widths, widths[1:])):
        layers += [P.Matvec(_w(r, a, b)), P.Bias(r.uniform(-0.1, 0.1, b))]
        if i < len(widths) - 2:
            layers.append(act(b))
    return layers


def _residual(r, n, w, out, blocks):
    layers = [P.Matvec(_w(r, n, w))]
    for _ in range(blocks):
        layers += [P.Save_State(0, w), P.LayerNorm(r.uniform(0.8, 1.2, w), r.uniform(-0.1, 0.1, w)),
                   P.Matvec(_w(r, w, w)), P.Gelu(w, True), P.Matvec(_w(r, w, w)), P.Bias(r.uniform(-0.1, 0.1, w)),
                   P.Binop_Add(0, w)]
    return layers + [P.Matvec(_w(r, w, out)), P.Softmax(out)]


def _projection(r, n, w):
    return [P.Save_State(1, n), P.Matvec(_w(r, n, w)), P.Sigmoid(w),
            P.Binop_Projection_Add(1, _w(r, n, w), r.uniform(-0.1, 0.1, w)), P.Binop_Concatenate(1, w, w + n, True),
            P.Matvec(_w(r, w + n, w)), P.Binop_Projection_Add(1, _w(r, n, w), r.uniform(-0.1, 0.1, w))]


CHAINS = {
    "odd_tiles": lambda r: _mlp(r, [20, 70, 130, 33], P.Tanh),       # 5, 9, 3 output tiles
    "few_tiles": lambda r: _mlp(r, [5, 40, 16, 40, 3], P.Relu),      # 3, 1, 3, 1
    "wide": lambda r: _mlp(r, [64, 250, 200, 64], P.Tanh),           # 16-bit: two column tiles
    "widest": lambda r: _mlp(r, [33, 520, 31], P.Silu),              # 16-bit: eight waves
    "residual": lambda r: _residual(r, 19, 70, 7, 2),
    "projection": lambda r: _projection(r, 21, 45),
}


@pytest.fixture(scope="module", autouse=True)
def _oracle_built():
    oracle.build()


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16", "f64"])
@pytest.mark.parametrize("chain", sorted(CHAINS))
def test_small_batch_and_main_kernels(cuda, chain, dtype):
    import torch

    if chain == "widest" and dtype in ("f32", "f64"):
        pytest.skip("wider than these types' fused kernels")
    layers = CHAINS[chain](np.random.default_rng(77))
    tdt = getattr(torch, TORCH_DT[dtype])
    small = P.create_inference_model(*layers, dtype=dtype, path="fused")
    main = P.create_inference_model(*layers, dtype=dtype, path="fused")
    A = P._abi
    A.check(A.lib().ponni_plan_device_params(main._plan, ctypes.byref(ctypes.c_void_p())))
    n_in, n_out = small.get_num_inputs(), small.get_num_outputs()
    for B, pad in [(1, 0), (16, 3), (33, 0), (64, 8), (515, 0)]:
        assert small.call_form(B) == "small"
        x = np.random.default_rng(B).standard_normal((n_in, B))
        xs = torch.zeros((n_in, B + pad), dtype=tdt, device="cuda:0")
        xs[:, :B] = torch.from_numpy(x).to(tdt)
        want = oracle.forward(layers, xs[:, :B].double().cpu().numpy(), ORACLE_MODE[dtype])
        for name in ("small", "main"):
            print(f"small batch: chain={chain} dtype={dtype} B={B} kernel={name}", flush=True)
            ys = torch.full((n_out, B + pad), float("nan"), dtype=tdt, device="cuda:0")
            stream = torch.cuda.current_stream().cuda_stream
            args = (xs.data_ptr(), xs.stride(0), ys.data_ptr(), ys.stride(0), B, stream)
            (small.forward_raw if name == "small" else main.forward_raw_no_alloc)(*args)
            torch.cuda.synchronize()
            assert torch.isnan(ys[:, B:].float()).all(), "kernel wrote past the batch"
            got = ys[:, :B].double().cpu().numpy()
            if dtype == "f32":
                check_f32(got, want)
            elif dtype == "f64":
                assert np.abs(got - want).max() <= 1e-12 * max(1.0, np.abs(want).max())
            else:
                check_half(got, want)


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("chain", ["few_tiles", "projection"])
def test_tiles_dealt_to_waves(cuda, chain, dtype):
    """Persistent kernels whose tiles go to waves (fp32 parameters in LDS,
    16-bit fragments in LDS): batches around one tile on every CU, around a
    wave on every SIMD, and of several passes with a ragged end, aligned and
    misaligned rows, on the main kernel."""
    import torch

    layers = CHAINS[chain](np.random.default_rng(78))
    tdt = getattr(torch, TORCH_DT[dtype])
    main = P.create_inference_model(*layers, dtype=dtype, path="fused")
    A = P._abi
    A.check(A.lib().ponni_plan_device_params(main._plan, ctypes.byref(ctypes.c_void_p())))
    n_in, n_out = main.get_num_inputs(), main.get_num_outputs()
    for B, pad in [(31, 1), (8_192, 0), (8_225, 7), (32_769, 7), (300_007, 1)]:
        print(f"tiles dealt to waves: chain={chain} dtype={dtype} B={B}", flush=True)
        x = np.random.default_rng(B).standard_normal((n_in, B))
        xs = torch.zeros((n_in, B + pad), dtype=tdt, device="cuda:0")
        xs[:, :B] = torch.from_numpy(x).to(tdt)
        ys = torch.full((n_out, B + pad), float("nan"), dtype=tdt, device="cuda:0")
        main.forward_raw_no_alloc(xs.data_ptr(), xs.stride(0), ys.data_ptr(), ys.stride(0), B,
                                  torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert torch.isnan(ys[:, B:].float()).all(), "kernel wrote past the batch"
        want = oracle.forward(layers, xs[:, :B].double().cpu().numpy(), ORACLE_MODE[dtype])
        (check_f32 if dtype == "f32" else check_half)(ys[:, :B].double().cpu().numpy(), want)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("chain", ["odd_tiles", "wide", "residual", "few_tiles"])
def test_half_rows_at_any_alignment_through_lds(cuda, chain, dtype):
    """Large batches of 16-bit rows that start anywhere (odd strides, column
    subviews): input through the blocks of 16 bytes around each row, outputs
    as unaligned vectors, against the oracle on a sample of columns that
    holds the batch's ends."""
    import torch

    layers = CHAINS[chain](np.random.default_rng(79))
    tdt = getattr(torch, TORCH_DT[dtype])
    m = P.create_inference_model(*layers, dtype=dtype, path="fused")
    n_in, n_out = m.get_num_inputs(), m.get_num_outputs()
    B = 150_001
    pick = np.concatenate([np.arange(70), np.random.default_rng(5).integers(70, B - 70, 1500), np.arange(B - 70, B)])
    x = np.random.default_rng(4).standard_normal((n_in, B)).astype(np.float32)
    xq = torch.from_numpy(x).to(tdt)
    want = oracle.forward(layers, xq[:, pick].double().numpy(), ORACLE_MODE[dtype])
    for off, pad in [(0, 0), (1, 0), (3, 4), (7, 7), (2, 5), (0, 1)]:
        print(f"rows at any alignment: chain={chain} dtype={dtype} off={off} pad={pad}", flush=True)
        xs = torch.zeros((n_in, off + B + pad), dtype=tdt, device="cuda:0")
        xs[:, off:off + B] = xq.cuda()
        ys = torch.full((n_out, off + B + pad), float("nan"), dtype=tdt, device="cuda:0")
        m.forward_batch_parallel(xs[:, off:off + B], ys[:, off:off + B])
        torch.cuda.synchronize()
        aligned = ((xs.data_ptr() + 2 * off) | (2 * xs.stride(0))) % 16 == 0
        assert m.call_form(B, 16 if aligned else 2) == ("main" if aligned else "any_rows")
        assert torch.isnan(ys[:, :off].float()).all() and torch.isnan(ys[:, off + B:].float()).all()
        got = ys[:, off:off + B].double().cpu().numpy()
        assert np.isfinite(got).all()
        check_half(got[:, pick], want)


@pytest.mark.parametrize("dtype", ["f32", "f16"])
def test_forms_first_used_by_several_threads(cuda, dtype):
    """One plan whose other kernels (small batches, misaligned rows) are first
    needed by several threads at once, each on a stream of its own: every
    thread's outputs are those of a plan used by one thread."""
    import threading

    import torch

    layers = CHAINS["odd_tiles"](np.random.default_rng(80))
    tdt = getattr(torch, TORCH_DT[dtype])
    one = P.create_inference_model(*layers, dtype=dtype, path="fused")
    shared = P.create_inference_model(*layers, dtype=dtype, path="fused")
    n_in = one.get_num_inputs()
    gen = torch.Generator(device="cuda").manual_seed(3)
    xs = [torch.randn((n_in, B), device="cuda", generator=gen).to(tdt) for B in (150_000, 64, 150_001, 515)]
    want = [one.forward_batch_parallel(x) for x in xs]
    shared.forward_batch_parallel(xs[0])  # parameters on the device, the main kernel loaded
    torch.cuda.synchronize()
    start, errors = threading.Barrier(len(xs)), []

    def work(i):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                start.wait(30)
                for j in [i, *range(len(xs))]:
                    y = shared.forward_batch_parallel(xs[j])
                    torch.cuda.current_stream().synchronize()
                    if not torch.equal(y, want[j]):
                        errors.append((i, j))
        except Exception as e:  # noqa: BLE001 (reported by the assertion below)
            errors.append((i, repr(e)))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(xs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert not any(t.is_alive() for t in threads) and not errors, errors


def test_one_tile_per_simd_costs_what_fewer_do(cuda):
    """Tiles dealt to waves spread over the SIMDs before any takes a second
    one, at every number of workgroups per CU (three here, where wave 0 of each
    was dealt to first and a SIMD took two of 32,768 columns' 1,024 tiles: 1.6 times
    the time of 16,384 columns)."""
    import torch

    r = np.random.default_rng(81)
    layers = [P.Matvec(_w(r, 9, 25))]
    for _ in range(2):
        layers += [P.Save_State(0, 25), P.LayerNorm(25), P.Matvec(_w(r, 25, 25)), P.Gelu(25, True),
                   P.Matvec(_w(r, 25, 25)), P.Binop_Add(0, 25)]
    m = P.create_inference_model(*layers, P.Matvec(_w(r, 25, 7)), dtype="f64", path="fused")
    A = P._abi
    A.check(A.lib().ponni_plan_device_params(m._plan, ctypes.byref(ctypes.c_void_p())))  # main kernel only
    us = {}
    for B in (16_384, 32_768):
        x = torch.randn((9, B), dtype=torch.float64, device="cuda:0")
        y = torch.empty((7, B), dtype=torch.float64, device="cuda:0")
        runs = []
        for _ in range(12):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(20):
                m.forward_raw_no_alloc(x.data_ptr(), B, y.data_ptr(), B, B, torch.cuda.current_stream().cuda_stream)
            b.record()
            torch.cuda.synchronize()
            runs.append(a.elapsed_time(b) * 50)
        us[B] = min(runs)
    print(f"one tile per SIMD: {us[32_768]:.1f} us, every other SIMD {us[16_384]:.1f}", flush=True)
    assert us[32_768] < 1.3 * us[16_384]


@pytest.mark.parametrize("dtype", ["f32", "f16", "f64"])
@pytest.mark.parametrize("chain", ["one", "three_tiles"])
def test_small_batch_kernel_in_place(cuda, chain, dtype):
    """y on x's own rows: every wave of a workgroup reads the columns that they
    all store.  One contraction (no exchange between the reads and the
    stores), and a first layer of three tiles, which leaves one of the four
    waves without one."""
    import torch

    r = np.random.default_rng(82)
    layers = {"one": lambda: [P.Matvec(_w(r, 100, 90)), P.Tanh(90)],
              "three_tiles": lambda: [P.Save_State(0, 48), P.Matvec(_w(r, 48, 48)), P.Relu(48),
                                      P.Binop_Projection_Add(0, _w(r, 48, 48), r.uniform(-0.1, 0.1, 48))]}[chain]()
    m = P.create_inference_model(*layers, dtype=dtype, path="fused")
    n_in, n_out = m.get_num_inputs(), m.get_num_outputs()
    for B in (16, 515, 4_096):
        assert m.call_form(B) == "small"
        print(f"in place: chain={chain} dtype={dtype} B={B}", flush=True)
        x = torch.randn((n_in, B), device="cuda:0", generator=torch.Generator("cuda:0").manual_seed(B))
        x = x.to(getattr(torch, TORCH_DT[dtype]))
        want = m.forward_batch_parallel(x)
        m.forward_batch_parallel(x, x[:n_out])
        torch.cuda.synchronize()
        assert torch.equal(x[:n_out], want)


_COMPILE_FORMS = """
import sys
import torch  # (its code generator, as in the process that uses the cache)
import numpy as np
import ponni_amd as P
r = np.random.default_rng(1)
m = P.create_inference_model(P.Matvec(r.uniform(-1, 1, (37, 75))), P.Tanh(75), P.Matvec(r.uniform(-1, 1, (75, 11))),
                             dtype="f16", path="fused")
print(m.call_form(64), m.call_form(300_001, 2), m.call_form(300_000, fp32_rows=True))
"""


def test_a_form_that_cannot_be_loaded_gives_way(cuda, tmp_path, monkeypatch):
    """A code cache whose objects for the small-batch and misaligned-row forms
    hold another kernel (here the main one's): those calls run on the main
    kernel, every time; fp32 rows are refused and infer_batch_half2's caller
    converts, as for a plan without that kernel."""
    import os
    import shutil
    import subprocess
    import sys

    import torch

    monkeypatch.setenv("PONNI_JIT_CACHE", str(tmp_path))
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    out = subprocess.run([sys.executable, "-c", _COMPILE_FORMS], cwd=root, capture_output=True, text=True, timeout=100,
                         env={**os.environ, "HIP_VISIBLE_DEVICES": "-1"})
    assert out.stdout.split() == ["small", "any_rows", "main"], out.stdout + out.stderr
    objects = {f: f.read_bytes() for f in tmp_path.iterdir() if f.suffix == ".co"}
    others = [f for f, code in objects.items() if any(s in code for s in (b"_split", b"_any", b"_io32"))]
    main = next(f for f in objects if f not in others)
    assert len(others) >= 3
    for f in others:
        shutil.copyfile(main, f)
    r = np.random.default_rng(1)
    layers = [P.Matvec(r.uniform(-1, 1, (37, 75))), P.Tanh(75), P.Matvec(r.uniform(-1, 1, (75, 11)))]
    m = P.create_inference_model(*layers, dtype="f16", path="fused")
    for B in (64, 300_001, 64):
        x = torch.randn((37, B), device="cuda:0", generator=torch.Generator("cuda:0").manual_seed(B)).half()
        y = m.forward_batch_parallel(x)
        torch.cuda.synchronize()
        assert torch.cuda.current_stream().query()
        check_half(y[:, :64].double().cpu().numpy(),
                   oracle.forward(layers, x[:, :64].double().cpu().numpy(), oracle.MODE_F16_OPERANDS))
        assert m.call_form(B, 2 if B % 8 else 16) == "main"
    x = torch.randn((37, 4096), device="cuda:0")
    for _ in range(2):
        assert not m.forward_fp32_rows(x, torch.empty((11, 4096), device="cuda:0"))


@pytest.mark.parametrize("chain", ["wide", "spilling"])
def test_small_batch_kernel_at_large_batches(cuda, chain):
    """Plans that run the small-batch kernel at every batch (fp32, wider than 448
    features, or spilling on the main kernel), with thousands of workgroups and
    a ragged last one: sampled columns, both ends among them, against the oracle."""
    import torch

    r = np.random.default_rng(83)
    layers = _mlp(r, [20, 464, 464, 60], P.Relu) if chain == "wide" else _residual(r, 12, 245, 35, 2)
    m = P.create_inference_model(*layers, dtype="f32", path="fused")
    B = 150_001
    assert m.call_form(B) == "small"
    pick = np.concatenate([np.arange(40), np.random.default_rng(6).integers(40, B - 40, 400), np.arange(B - 40, B)])
    x = torch.randn((m.get_num_inputs(), B), device="cuda:0", generator=torch.Generator("cuda:0").manual_seed(7))
    ys = torch.full((m.get_num_outputs(), B + 3), float("nan"), device="cuda:0")
    m.forward_batch_parallel(x, ys[:, :B])
    torch.cuda.synchronize()
    assert torch.isnan(ys[:, B:]).all() and torch.isfinite(ys[:, :B]).all()
    check_f32(ys[:, pick].double().cpu().numpy(), oracle.forward(layers, x[:, pick].double().cpu().numpy()))
