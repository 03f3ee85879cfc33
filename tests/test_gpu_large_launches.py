"""Calls whose threads number 2^32 or more: a grid of that size is cut off by the runtime without
an error, so they take several launches.  Values are constants or one-line sums, on 20 to 80 GB."""

import sys

import pytest
import torch

from gstools_amd.krige import krige_sum_device

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _memory():
    torch.cuda.empty_cache()
    yield
    torch.cuda.empty_cache()


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def _full(shape, value):
    return torch.full(shape, value, dtype=torch.float64, device="cuda")


@pytest.mark.parametrize("p", [2**31 + 1, 2**31 + 2])
def test_kriging_field_of_many_points(p):
    _say(f"krige field P={p}")
    field = krige_sum_device(_full((1, 1), 1.0), _full((1, p), 2.0), _full((1,), 1.5), variance=False)
    assert bool((field == 3.0).all())
