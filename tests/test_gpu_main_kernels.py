"""The main kernels of FUSED plans on the random, non-finite and op-graph tests
of the other files.

Their batches are small, and ponni_forward runs most of them on the small-batch
kernel.  Here every FUSED plan is put on the device by ponni_plan_device_params,
which loads its main kernel only, and called through the allocation-free entry,
which loads nothing; half-precision graphs convert around it."""
import ctypes

import pytest

import oracle
import ponni_amd as P
from tests import test_gpu_fuzz as fuzz
from tests import test_gpu_graph_ops as graph_ops
from tests import test_gpu_parity as parity

pytestmark = pytest.mark.gpu
DTYPES = ["f32", "f16", "bf16", "f64"]


@pytest.fixture(scope="module", autouse=True)
def _oracle_built():
    oracle.build()


@pytest.fixture(autouse=True)
def main_kernels(monkeypatch):
    """Calls of FUSED plans through ponni_forward_no_alloc; the list of them."""
    ordinary, calls = P.Inference.forward_raw, []

    def forward_raw(self, x_ptr, ld_in, y_ptr, ld_out, batch, stream=0):
        if self.path != "fused":
            return ordinary(self, x_ptr, ld_in, y_ptr, ld_out, batch, stream)
        A = P._abi
        A.check(A.lib().ponni_plan_device_params(self._plan, ctypes.byref(ctypes.c_void_p())))
        calls.append(batch)
        return self.forward_raw_no_alloc(x_ptr, ld_in, y_ptr, ld_out, batch, stream)

    monkeypatch.setattr(P.Inference, "forward_raw", forward_raw)
    monkeypatch.setattr(P.Inference, "forward_fp32_rows", lambda self, x, y: False)
    return calls


@pytest.mark.parametrize("seed", range(10))
def test_random_chains(cuda, main_kernels, seed):
    parity.test_random_chains(cuda, seed, "fused")
    assert main_kernels


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("seed", range(4))
def test_random_chains_reduced_precision(cuda, main_kernels, dtype, seed):
    parity.test_random_chains_reduced_precision_fused(cuda, dtype, seed)
    assert main_kernels


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("chain", sorted(c for c in parity.NONFINITE_CHAINS if parity.NONFINITE_CHAINS[c][1]))
def test_non_finite_inputs(cuda, main_kernels, chain, dtype):
    parity.test_non_finite_inputs(cuda, chain, "fused", dtype)
    assert main_kernels


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("chain", sorted(parity.PADDED_DENSE_CHAINS))
def test_infinities_through_padded_dense_layers(cuda, main_kernels, chain, dtype):
    parity.test_infinities_through_padded_dense_layers(cuda, chain, "fused", dtype)
    assert main_kernels


@pytest.mark.parametrize("dtype", ["f32", "f16", "f64"])
@pytest.mark.parametrize("after", [True, False])
def test_concatenation_any_lead_width(cuda, main_kernels, after, dtype):
    parity.test_concatenation_any_lead_width_fused(cuda, after, dtype)
    assert main_kernels


@pytest.mark.parametrize("group", range(fuzz.GROUPS))
def test_random_cases(cuda, main_kernels, group):
    fuzz.test_random_cases(cuda, group)
    assert main_kernels


@pytest.mark.parametrize("group", range(2))
def test_random_wide_cases(cuda, main_kernels, group):
    fuzz.test_random_wide_cases(cuda, group)
    assert main_kernels


@pytest.mark.parametrize("group", range(2))
def test_random_non_finite_cases(cuda, main_kernels, group):
    fuzz.test_random_non_finite_cases(cuda, group)
    assert main_kernels


@pytest.mark.parametrize("dtype", ["f32", "f16"])
@pytest.mark.parametrize("seed", range(6))
def test_op_graphs(cuda, main_kernels, seed, dtype):
    graph_ops.test_op_graphs_on_gpu(cuda, seed, "fused", dtype)
    assert main_kernels


@pytest.mark.parametrize("dtype", ["f32", "f16"])
@pytest.mark.parametrize("n", [12, 16])
def test_reductions_of_non_finite_inputs(cuda, main_kernels, n, dtype):
    graph_ops.test_reductions_of_non_finite_inputs(cuda, n, "fused", dtype)
    assert main_kernels
