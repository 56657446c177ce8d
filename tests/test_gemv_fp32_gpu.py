"""The fp32 GEMV's own plan past 4096 outputs takes the cached-load twin of its
configuration: the same sums in the same order, so the same bits as that
configuration named."""
import pytest
import torch

from conftest import say
from spmv_decode_amd import _lib
from test_gemv_gpu import make_case, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1024, 4096), (1024, 4224), (2048, 16384), (1000, 16512)], ids=str)
def test_fp32_plan_keeps_its_bits(gpu, shape):
    K, h = shape
    x, md, mi = make_case(K, h, 4, 8, seed=K + h, dtype=torch.float32)
    p = _lib.plan(h, md.shape[0], 4, 8)
    say(f"fp32 gemv {shape} plan {p}")
    assert torch.equal(run(x, md, mi, 4, 8), run(x, md, mi, 4, 8, config_id=p["config_id"], splits=p["splits"]))


@pytest.mark.parametrize("shape", [(2048, 8192), (1024, 8192), (2048, 8064), (512, 28672), (512, 28800)], ids=str)
def test_fp32_plan_keeps_its_bits_on_both_sides_of_the_cached_loads(gpu, shape):
    """One whole round of workgroups over 1024 and 512 compressed columns, 28672 outputs and one tile more."""
    test_fp32_plan_keeps_its_bits(gpu, shape)
