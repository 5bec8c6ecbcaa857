"""The profile summaries name each kernel's class as the engine's profiler does."""
import pytest

from mignon_ai_amd.profsum import kernel_class


@pytest.mark.parametrize("kernel,cls", [
    ("void mg::(anonymous namespace)::gemm_c2_kernel<false>(mg::GemmArgs)", "gemm_i8"),
    ("void mg::(anonymous namespace)::gemm_c2_kernel<true>(mg::GemmArgs)", "gemm_i8"),
    ("mg::(anonymous namespace)::gemm_thin_kernel(mg::GemmArgs)", "gemm_i8"),
    ("void mg::(anonymous namespace)::gemm_slab_kernel<6, 0, true, 1>(mg::GemmArgs, int, int)", "gemm_logits"),
    ("void mg::(anonymous namespace)::seq_kernel<2, 4, 2, false>(mg::SeqArgs)", "sequence_body"),
    ("void mg::(anonymous namespace)::export_kv_packed_dpp_kernel<8>(int)", "state_export"),
])
def test_kernel_class(kernel, cls):
    assert kernel_class(kernel) == cls
