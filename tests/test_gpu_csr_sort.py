"""The CSR of unsorted keys (ictc_csr_build) is exactly the stable sort by key, on both sides of every rule."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,N", [(1, 1), (63, 3), (1024, 255), (1025, 254), (4097, 10), (5000, 256), (70001, 1359),
                                 (20000, 65535), (3000, 65536), (262144, 4096), (262145, 4096)])
def test_csr_is_a_stable_sort(device, E, N):
    """Both digit passes, tile and stretch edges, ids out of range (last), and the library sort's side of the rule."""
    from ictc_o3.ops.tensor_product import Csr
    g = torch.Generator().manual_seed(E)
    keys = torch.randint(0, N, (E,), generator=g)
    if E > 10:
        keys[::7] = N - 1                     # a long segment
        keys[3], keys[5] = -2, N + 9
    k = torch.where((keys < 0) | (keys >= N), torch.full_like(keys, N), keys)
    csr = Csr(keys.to(device), N)
    assert torch.equal(csr.order[:E].long().cpu(), torch.argsort(k, stable=True))
    want = torch.cat([torch.searchsorted(k.sort().values, torch.arange(N + 1)), torch.tensor([E])])
    assert torch.equal(csr.ptr.long().cpu(), want)


@pytest.mark.parametrize("largest,E,N", [((262145, 4096), 262144, 4096), ((262145, 4096), 1000, 100),
                                         ((1000, 65536), 1000, 4096), ((1000, 65536), 1000, 100),
                                         ((1000, 65536), 1, 65536), ((5000, 4096), 4096, 4096),
                                         ((200001, 65535), 200000, 65535)])
def test_workspace_of_a_larger_list(device, largest, E, N):
    from ictc_o3 import _native as nat
    nbytes = int(nat.lib().ictc_csr_workspace_bytes(*largest))
    ws = torch.empty(nbytes, dtype=torch.uint8, device=device)
    keys = torch.randint(0, N, (E,), device=device, generator=torch.Generator(device=device).manual_seed(E))
    ptr = torch.empty(N + 2, dtype=torch.int32, device=device)
    order = torch.empty(E, dtype=torch.int32, device=device)
    nat.call("ictc_csr_build", nat.ptr(keys), E, N, nat.ptr(ptr), nat.ptr(order), nat.ptr(ws), nbytes,
             nat.stream_of(keys))
    assert torch.equal(order.long(), torch.argsort(keys, stable=True))


def _bytes(E):
    """The counting sort's storage (its counts in whole groups of 4,096, keys and ids of both passes)."""
    tiles = (E + 1023) // 1024
    return 4 * 4096 * ((256 * tiles + 4095) // 4096) + (12 * E + 255) // 256 * 256


@pytest.mark.parametrize("E,N", [(4096, 300), (4097, 300), (1, 256), (200000, 65535), (200001, 65535), (170000, 40000)])
def test_either_sort_gives_the_stable_order(device, E, N):
    """On both sides of the rule that chooses the sort; and with room for the counting sort alone, which it then is."""
    from ictc_o3 import _native as nat
    keys = torch.randint(0, N, (E,), device=device, generator=torch.Generator(device=device).manual_seed(E))
    want = torch.argsort(keys, stable=True)
    for nbytes in (int(nat.lib().ictc_csr_workspace_bytes(E, N)), _bytes(E)):
        ws = torch.empty(nbytes, dtype=torch.uint8, device=device)
        ptr = torch.empty(N + 2, dtype=torch.int32, device=device)
        order = torch.empty(E, dtype=torch.int32, device=device)
        nat.call("ictc_csr_build", nat.ptr(keys), E, N, nat.ptr(ptr), nat.ptr(order), nat.ptr(ws), nbytes,
                 nat.stream_of(keys))
        assert torch.equal(order.long(), want)
