"""The forward's shape tests once more with the kernel left to the library, as every operator leaves it: a call that names
one keeps its keys whole, and so never runs the kernels whose halves share them out."""

import pytest
from test_fwd_gpu import (  # noqa: F401
    pytestmark,
    test_config2_bf16_causal_mha,
    test_mfma_forward_masked_head_dim_64,
    test_mfma_forward_matrix,
    test_mfma_forward_narrow_head_dims,
    test_mfma_forward_padding_masks_with_holes_and_dead_batches,
    test_mfma_forward_rows_whose_first_keys_are_masked,
    test_mfma_forward_value_rows_narrower_than_keys,
    test_mfma_forward_with_bias_and_masks,
    test_mfma_forward_with_kv_lens,
    test_noncontiguous_inputs_keep_query_layout,
    test_short_queries_with_grouped_heads,
    test_softmax_reference_tracking_under_stress,
)


class _Unnamed:
    """The package, with forwards that name no kernel."""

    def __init__(self, amd):
        self._amd = amd

    def __getattr__(self, name):
        return getattr(self._amd, name)

    def sdpa_forward(self, *args, force_kernel=0, **kw):
        return self._amd.sdpa_forward(*args, **kw)


@pytest.fixture(scope="module")
def amd(gpu_device):
    import torch_neuronx_amd as amd

    return _Unnamed(amd)
