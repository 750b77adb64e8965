"""Sorting of a tile's list at the lengths where the number of runs, of entries per lane or the kernel changes, bit for bit
against the oracle: one tile, every surfel in it, depths with many values in common (the surfel's number then decides)."""
import numpy as np
import pytest
import torch

from util import npy

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n', [1, 2, 63, 64, 65, 127, 128, 129, 192, 193, 255, 256, 257, 449, 511, 512, 513, 1000, 1024, 1025,
                               1536, 1601, 2047, 2048, 2049])
@pytest.mark.parametrize('depths', ['equal', 'few', 'rising', 'falling', 'random'])
def test_list_of_one_tile(n, depths, device, oracle_mod):
    from fast_sp_gs_amd._C import get_C_function
    print(f'[tile sort] n={n} {depths}', flush=True)
    g = torch.Generator().manual_seed(n)
    dep = {'equal': torch.ones(n), 'few': torch.randint(1, 4, (n,), generator=g).float(), 'rising': torch.arange(1.0, n + 1),
           'falling': torch.arange(float(n), 0.0, -1.0), 'random': torch.rand(n, generator=g) + 0.5}[depths]
    m2 = torch.full((n, 2), 8.0)
    radii, touched = torch.full((n,), 3, dtype=torch.int32), torch.ones(n, dtype=torch.int32)
    ranges, pl, keys = get_C_function('GS_prepare')(16, 16, m2.to(device), dep.to(device), radii.to(device),
                                                    touched.to(device), False, return_keys=True)[:3]
    want_ranges, want_pl, want_keys = oracle_mod.prepare(16, 16, npy(m2), npy(dep), npy(radii), npy(touched), return_keys=True)
    assert want_pl.size == n
    assert np.array_equal(npy(ranges), want_ranges) and np.array_equal(npy(pl), want_pl) and np.array_equal(npy(keys), want_keys)


@pytest.mark.parametrize('n', [1, 2, 65, 255, 256, 257, 512, 513, 1024, 1025, 1999, 2048])
@pytest.mark.parametrize('depths', ['shells', 'outlier', 'signs', 'ties'])
def test_list_of_one_tile_by_buckets(n, depths, device, oracle_mod):
    """Depths that fill few buckets (two thin shells, one far value) or span all bit patterns, and buckets with ties."""
    from fast_sp_gs_amd._C import get_C_function
    print(f'[tile sort] n={n} {depths}', flush=True)
    g = torch.Generator().manual_seed(n)
    r = torch.rand(n, generator=g)
    far = r + 1.0
    far[n // 2] = 3e38
    dep = {'shells': torch.randint(1, 3, (n,), generator=g).float() + 1e-3 * r, 'outlier': far,
           'signs': torch.randn(n, generator=g) * 10.0 ** torch.randint(-30, 30, (n,), generator=g),
           'ties': (r * n / 4).floor() + 1.0}[depths].float()
    m2 = torch.full((n, 2), 8.0)
    radii, touched = torch.full((n,), 3, dtype=torch.int32), torch.ones(n, dtype=torch.int32)
    ranges, pl, keys = get_C_function('GS_prepare')(16, 16, m2.to(device), dep.to(device), radii.to(device),
                                                    touched.to(device), False, return_keys=True)[:3]
    want_ranges, want_pl, want_keys = oracle_mod.prepare(16, 16, npy(m2), npy(dep), npy(radii), npy(touched), return_keys=True)
    assert np.array_equal(npy(ranges), want_ranges) and np.array_equal(npy(pl), want_pl) and np.array_equal(npy(keys), want_keys)


@pytest.mark.parametrize('n', [2, 33, 200, 256, 257, 700, 1025, 2048])
@pytest.mark.parametrize('depths', ['one', 'two', 'one of many', 'shells'])
def test_equal_depths_in_one_of_two_tiles(n, depths, device, oracle_mod):
    """Equal depths are put in order by the surfels' numbers: spread over the tile's span of numbers, or in two clumps of it (the
    cut by numbers then fills a few parts only). `one of many`: one bucket of many depths holds one depth a hundred times;
    `shells`: buckets of several depths beside buckets of one."""
    from fast_sp_gs_amd._C import get_C_function
    print(f'[tile sort] n={n} equal depths: {depths}', flush=True)
    g = torch.Generator().manual_seed(n)
    for clumped in (False, True):
        P = 20 * n
        here = torch.zeros(P, dtype=torch.bool)
        here[torch.cat([torch.arange(n // 2), P - 1 - torch.arange(n - n // 2)]) if clumped else torch.randperm(P, generator=g)[:n]] = True
        r = torch.rand(P, generator=g)
        dep = {'one': torch.full((P,), 3.0), 'two': torch.randint(3, 5, (P,), generator=g).float(),
               'one of many': torch.where(r < 0.3, torch.full((P,), 2.0), 1.0 + 4.0 * r),
               'shells': torch.where(r < 0.5, torch.full((P,), 3.0), 4.0 + 1e-4 * r)}[depths]
        m2 = torch.stack([torch.where(here, 8.0, 24.0), torch.full((P,), 8.0)], 1).contiguous()
        keep = here | (torch.rand(P, generator=g) < 0.02)  # a few in the other tile
        radii, touched = torch.where(keep, 3, 0).int(), keep.int()
        ranges, pl, keys = get_C_function('GS_prepare')(32, 16, m2.to(device), dep.to(device), radii.to(device),
                                                        touched.to(device), False, return_keys=True)[:3]
        want = oracle_mod.prepare(32, 16, npy(m2), npy(dep), npy(radii), npy(touched), return_keys=True)
        assert want[0][0, 1] - want[0][0, 0] == n
        for a, b in zip((ranges, pl, keys), want):
            assert np.array_equal(npy(a), b)


@pytest.mark.parametrize('n', [2049, 4095, 4096, 4097, 8192, 8193, 16383, 16384, 16385, 32769, 50_000])
@pytest.mark.parametrize('depths', ['random', 'equal', 'ties', 'shells', 'outlier', 'signs'])
def test_long_list_of_one_tile(n, depths, device, oracle_mod):
    """Lists that the 1024-lane blocks sort: by buckets in LDS, by groups of buckets above 16 384 entries, and by the network where
    too many entries share a bucket (`equal`, `outlier`, and `shells` at the larger sizes)."""
    from fast_sp_gs_amd._C import get_C_function
    print(f'[tile sort] n={n} {depths}', flush=True)
    g = torch.Generator().manual_seed(n)
    r = torch.rand(n, generator=g)
    far = r + 1.0
    far[n // 2] = 3e38
    dep = {'random': r * 10.0 + 0.5, 'equal': torch.ones(n), 'ties': (r * n / 4).floor() + 1.0,
           'shells': torch.randint(1, 3, (n,), generator=g).float() + 1e-3 * r, 'outlier': far,
           'signs': torch.randn(n, generator=g) * 10.0 ** torch.randint(-30, 30, (n,), generator=g)}[depths].float()
    m2 = torch.full((n, 2), 8.0)
    radii, touched = torch.full((n,), 3, dtype=torch.int32), torch.ones(n, dtype=torch.int32)
    ranges, pl, keys = get_C_function('GS_prepare')(16, 16, m2.to(device), dep.to(device), radii.to(device),
                                                    touched.to(device), False, return_keys=True)[:3]
    want_ranges, want_pl, want_keys = oracle_mod.prepare(16, 16, npy(m2), npy(dep), npy(radii), npy(touched), return_keys=True)
    assert np.array_equal(npy(ranges), want_ranges) and np.array_equal(npy(pl), want_pl) and np.array_equal(npy(keys), want_keys)
