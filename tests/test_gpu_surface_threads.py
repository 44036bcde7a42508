"""The surface kernel's two workgroup sizes at the line between them: 9 facet
blocks (the last one partly filled) by 56 shots (504 workgroups of 1024
threads) and by 57 (513 of 256), against the FP64 oracle.

Tolerance: helpers.compare_traces; both sizes sum the same FP32 terms in FP64
or fixed-point windows."""
import pytest

from europaraypaths_amd._abi import ERP_RUN_DETERMINISTIC
from tests.test_gpu_spectral_stages import check, scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flags", [0, ERP_RUN_DETERMINISTIC])
@pytest.mark.parametrize("spec", [False, True])
@pytest.mark.parametrize("ns", [56, 57])
def test_both_workgroup_sizes(gpu_ctx, ns, spec, flags):
    over = dict(specular=True, convolution=True, convolution_linear=True,
                rerad_funct=0) if spec else {}
    check(gpu_ctx, *scene(700, nx=100, ny=184, ns=ns, targets=2, **over), flags=flags)
