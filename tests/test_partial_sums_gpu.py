"""Partial sums of the filter gradients shared by several threads: few outputs, many strips."""
import pytest
import torch

import test_spatial_norm_gpu as spatial_norm
from ddf_testlib import check_against_oracle, random_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dtype', [torch.float64, torch.float32, torch.float16])
@pytest.mark.parametrize('shape', [
    (1, 1, 3100, 40),     # the most threads per output, stretches of unequal length
    (1, 3, 97, 40), (2, 5, 193, 64), (1, 40, 200, 41),
    (1, 24, 48, 128),     # with the sum over channel ranges in the same launch
])
def test_many_strips(shape, dtype):
    case = random_case(*shape, 3, 1, dtype, seed=7)
    check_against_oracle(*case, 3, 1, 1, 'mul', '', what='many strips')


@pytest.mark.parametrize('shape,k', [((1, 4, 300, 40), 3), ((1, 4, 90, 40), 5)])
def test_many_strips_behind_the_normalisation(shape, k):
    spatial_norm.test_backward_spatial_norm_through_the_c_abi(shape, k, 1, 1, 'mul', torch.float32, 1, True)
