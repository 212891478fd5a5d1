"""Into how many parts the latent attention divides its keys, against times that were measured."""
import pytest

from yalis_amd.ops.hip import HipOps

# heads, latent, cached, new tokens, requests; us by parts (one MI355X, a latent's rows 32 or 64 longer)
MEASURED = [
    (16, 512, 0, 512, 1, {1: 49.7, 2: 46.9, 4: 68.0, 8: 111.0}),
    (16, 512, 1536, 512, 1, {1: 139.2, 2: 92.6, 4: 113.9, 8: 157.1}),
    (16, 512, 1000, 1, 8, {1: 49.1, 2: 32.1, 4: 21.9, 8: 18.2, 16: 15.7, 32: 17.3}),
    (16, 512, 500, 1, 64, {1: 33.0, 2: 27.8, 4: 27.7, 8: 39.5, 16: 57.7}),
    (32, 256, 1536, 512, 1, {1: 94.1, 2: 118.9, 4: 141.9, 8: 194.8}),
    (16, 256, 4000, 1, 8, {1: 122.2, 2: 68.7, 4: 40.3, 8: 25.9, 16: 19.6, 32: 17.9}),
    (16, 256, 0, 100, 8, {1: 17.9, 2: 37.7}),
    (8, 128, 0, 2048, 1, {1: 70.0, 2: 69.6}),
    (16, 128, 3000, 1, 2, {1: 79.3, 2: 44.9, 4: 26.4, 8: 16.8, 16: 12.7, 32: 11.9, 64: 14.3}),
    (4, 64, 0, 512, 1, {1: 17.5, 2: 14.4, 4: 11.5, 8: 10.6, 16: 13.2, 32: 19.6}),
    (16, 64, 0, 512, 1, {1: 17.9, 2: 19.4, 4: 20.4, 8: 27.4, 16: 38.9}),
    (16, 64, 1000, 1, 1, {1: 24.1, 2: 16.9, 4: 11.5, 8: 9.1, 16: 8.5, 32: 9.2}),
    (16, 64, 0, 33, 1, {1: 5.3, 2: 8.3, 4: 8.5, 8: 8.9}),
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
