"""Into how many parts the latent attention divides its keys, against times that were measured."""
import pytest

from yalis_amd.ops.hip import HipOps

# heads, latent, cached, new tokens, requests; us by parts (one MI355X, a latent's rows 32 or 64 longer)
MEASURED = [
    (16, 512, 0, 512, 1, {1: 50.9, 2: 48.8, 4: 68.3, 8: 111.0}),
    (16, 512, 1536, 512, 1, {1: 140.4, 2: 93.7, 4: 113.7, 8: 158.2}),
    (16, 512, 1000, 1, 8, {1: 50.4, 2: 33.3, 4: 23.1, 8: 18.4, 16: 18.3, 32: 18.9}),
    (16, 512, 500, 1, 64, {1: 34.2, 2: 28.9, 4: 29.1, 8: 41.1, 16: 62.9}),
    (32, 256, 1536, 512, 1, {1: 93.8, 2: 111.0, 4: 136.6, 8: 193.0}),
    (16, 256, 4000, 1, 8, {1: 120.4, 2: 67.7, 4: 40.0, 8: 26.2, 16: 20.0, 32: 18.7}),
    (16, 256, 0, 100, 8, {1: 19.0, 2: 38.8}),
    (8, 128, 0, 2048, 1, {1: 70.2, 2: 63.2}),
    (16, 128, 3000, 1, 2, {1: 73.5, 2: 42.5, 4: 25.3, 8: 16.7, 16: 12.9, 32: 12.5, 64: 14.7}),
    (4, 64, 0, 512, 1, {1: 18.6, 2: 15.3, 4: 12.4, 8: 11.2, 16: 16.5, 32: 24.2}),
    (16, 64, 0, 512, 1, {1: 19.0, 2: 20.4, 4: 23.8, 8: 32.7, 16: 49.5}),
    (16, 64, 1000, 1, 1, {1: 28.8, 2: 19.6, 4: 13.2, 8: 10.1, 16: 9.4, 32: 10.3}),
    (16, 64, 0, 33, 1, {1: 6.4, 2: 9.4, 4: 9.6, 8: 10.0}),
]


@pytest.mark.parametrize("heads,latent,cached,new,requests,us", MEASURED)
def test_keys_are_divided_as_measured(heads, latent, cached, new, requests, us):
    """No more than an eighth slower than the best of the numbers that were tried."""
    a_tile = max(1, 64 // heads)
    parts = HipOps.latent_attention_splits(requests * -(-new // a_tile), heads, cached + new, requests * new, latent)
    assert us[parts] <= 1.125 * min(us.values()), parts


@pytest.mark.parametrize("keys", [1, 31, 32, 33, 64, 65])
def test_a_part_has_keys(keys):
    assert HipOps.latent_attention_splits(1, 16, keys, 1, 512) <= -(-keys // 32)


@pytest.mark.parametrize("heads", [1, 4, 16, 48, 64, 65, 128])
@pytest.mark.parametrize("latent", [64, 128, 256, 512])
def test_decode_steps_fit_the_scratch_that_captures_reserve(heads, latent):
    """A captured step may not grow its scratch, and 1 << 24 floats are reserved: a division never makes 512 workgroups (beyond 256 it wins
    nothing), each of which leaves 64 columns of the latent and two numbers."""
    for requests in list(range(1, 260)) + [300, 511, 512, 1024]:
        for keys in (256, 512, 1024, 4096, 16384, 131072, 1 << 20):
            parts = HipOps.latent_attention_splits(requests, heads, keys, requests, latent)
            assert parts == 1 or requests * -(-heads // 64) * parts * 64 * (latent + 2) <= 1 << 24
