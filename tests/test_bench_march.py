"""bench.py names the march that its plan takes."""

from types import SimpleNamespace

import pytest

import bench


@pytest.mark.parametrize("block,marches,name", [
    (256, (0, 128), "k_shoot_pair<false,256>"),
    (64, (0, 128), "k_shoot_pair<false,64>"),
    (128, (1, 0), "k_shoot<1,false,true,128>"),
    (256, (2, 46), "k_shoot_pair<false,256> and k_shoot<1,false,true,256>"),
])
def test_the_march_is_named_by_the_plan(block, marches, name):
    fb = SimpleNamespace(tuning={"shoot_block": block}, plan=SimpleNamespace(marches=lambda: marches))
    assert bench.march_kernel(fb) == name
