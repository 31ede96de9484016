"""The prefix broadcast in the sizes where a thread serves up to eight destinations (more than 16 workgroups per compute unit with
one destination each), next to the sizes of test_gpu_broadcast.py, most of which have a workgroup per destination."""
import pytest

from test_gpu_broadcast import test_every_layer_and_destination as every_layer_and_destination

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kv_bits,Hk,L,G,src,dst,T", [
    (4, 8, 16, 19, 5, (0, 19), 64),     # 18 destinations: two groups of eight and one of two, source among them
    (2, 1, 40, 34, 33, (0, 33), 33),    # norm rows of two bytes: the narrow copy
    (0, 8, 28, 10, 0, (1, 10), 200),    # fp16: a group of eight and one of one
    (4, 8, 28, 8, 3, (0, 8), 512),      # seven destinations: less than a group
    (4, 8, 1, 18, 0, (1, 18), 4096),    # one layer, just past the line
])
def test_groups_of_destinations(kv_bits, Hk, L, G, src, dst, T):
    every_layer_and_destination(kv_bits, Hk, L, G, src, dst, T)
