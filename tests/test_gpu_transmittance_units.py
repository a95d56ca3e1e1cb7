"""The batched transmittance queries' work split: an estimate depends on its ray, sample and seed alone, so results must
be the same bits however many rays share the call, in whatever launches the units go, and from whichever stream."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ESTIMATORS = ["delta", "ratio", "residual_ratio", "decomposition"]


@pytest.fixture(scope="module")
def cloud(vpt):
    vpt.generate_fbm_cloud(48, 40, 44, seed=3)
    vpt.set_vpt_mode(0)
    vpt.set_grid_interpolation_type(1)
    vpt.set_extinction_base([1.0, 1.0, 1.0])
    vpt.set_extinction_scale(200.0)
    return vpt


def _rays(n):
    import torch

    g = torch.Generator().manual_seed(1)
    o = torch.randn((n, 3), generator=g)
    o = 0.8 * o / o.norm(dim=1, keepdim=True)
    d = (torch.rand((n, 3), generator=g) - 0.5) * 0.6 - o
    return o.cuda(), (d / d.norm(dim=1, keepdim=True)).cuda()


@pytest.mark.parametrize("sparse,interpolation", [(False, 1), (True, 1), (True, 0), (True, 2)])
@pytest.mark.parametrize("estimator", ESTIMATORS)
def test_batch_size_does_not_matter(cloud, estimator, sparse, interpolation):
    print(f"case: transmittance units {estimator} sparse={sparse} interpolation={interpolation}", flush=True)
    cloud.set_use_sparse_grid(sparse)
    cloud.set_grid_interpolation_type(interpolation)
    o, d = _rays(3001)
    for samples in (1, 2, 7):
        mean, m2 = cloud.transmittance_batch(estimator, o, d, None, samples, 5)
        for n in (1, 63, 65, 1000):
            a, b = cloud.transmittance_batch(estimator, o[:n], d[:n], None, samples, 5)
            assert bool((a == mean[:n]).all()) and bool((b == m2[:n]).all())
        host, host2 = cloud.transmittance_batch(estimator, o.cpu().numpy(), d.cpu().numpy(), None, samples, 5)
        assert np.array_equal(host, mean.cpu().numpy()) and np.array_equal(host2, m2.cpu().numpy())


def test_many_samples_take_several_launches(cloud):
    """3 x 2^25 estimates go in launches of two rays; 2^26 + 3 of one ray in two launches whose sums continue."""
    print("case: transmittance units in several launches", flush=True)
    cloud.set_use_sparse_grid(False)
    cloud.set_grid_interpolation_type(1)
    o, d = _rays(3)
    mean, m2 = cloud.transmittance_batch("delta", o, d, None, 1 << 25, 2)
    one, one2 = cloud.transmittance_batch("delta", o[:1], d[:1], None, 1 << 25, 2)
    assert float(one[0]) == float(mean[0]) and float(one2[0]) == float(m2[0])
    n = (1 << 26) + 3
    long, _ = cloud.transmittance_batch("delta", o[:1], d[:1], None, n, 2)
    # the first half's and the whole's mean differ by the second half's sampling error: 5 sigma of a 0/1 estimate
    p = float(one[0])
    assert abs(float(long[0]) - p) <= 5.0 * np.sqrt(max(p * (1.0 - p), 1e-9) / (1 << 25)) + 1e-6


def test_streams_share_the_estimates_buffer(cloud):
    print("case: transmittance units on two streams", flush=True)
    import torch

    cloud.set_use_sparse_grid(False)
    o, d = _rays(20000)
    ref = [cloud.transmittance_batch("ratio", o, d, None, 4, s) for s in (1, 2)]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    for _ in range(5):
        got = []
        for k, st in enumerate(streams):
            with torch.cuda.stream(st):
                got.append(cloud.transmittance_batch("ratio", o, d, None, 4, k + 1))
        torch.cuda.synchronize()
        for (a, a2), (b, b2) in zip(ref, got):
            assert bool((a == b).all()) and bool((a2 == b2).all())
