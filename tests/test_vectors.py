"""Weights with one diagonal factor and nothing else: update and application in one launch each (csrc/elem.hip,
vec_update_kernel and vec_apply_kernel) up to 16384 elements, a launch per stage above."""
import pytest
import torch

from tests.test_gpu_parity import assert_fp32, run_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(2, 63), (1023, 1024, 1025), (1, 1531, 16384), (16385,)])
@pytest.mark.parametrize("gdt", [torch.float32, torch.bfloat16])
def test_vectors_with_a_diagonal_factor(sizes, gdt):
    """Against the float64 oracle at the fp32 bar, sizes around the workgroup's 1024 threads and the one-launch limit, as
    columns and as rows; equal sizes share a launch."""
    shapes = [s for n in sizes for s in ((n,), (n, 1), (1, n))]
    worst, base = run_pair(shapes, steps=3, skew=1.0, gdt=gdt, grad_eps=float(torch.finfo(gdt).eps))
    assert_fp32(worst, base)
