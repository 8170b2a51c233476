"""The choice between the two attention paths of a long forward, at shapes where
one of them was measured at least a quarter faster."""
import pytest

from versenext_amd.model import chain_pays


# (B, H, Hkv, d, window, n, cached), us of the chain kernel, us of the chunks
@pytest.mark.parametrize("shape,chain,chunks", [
    ((1, 16, 8, 64, 1024, 65, 2000), 28, 35), ((1, 16, 8, 64, 1024, 130, 2000), 27, 58),
    ((1, 16, 8, 64, 16384, 512, 4000), 64, 197), ((1, 16, 8, 64, 16384, 65, 8000), 102, 49),
    ((1, 8, 8, 128, 16384, 65, 8000), 178, 58), ((2, 16, 8, 64, 16384, 65, 4000), 56, 41),
    ((1, 8, 8, 128, 4096, 65, 4000), 97, 48)])
def test_the_faster_path(shape, chain, chunks):
    assert chain_pays(*shape, 256) == (chain < chunks)


def test_every_shape_has_an_answer():
    for d in (64, 128):
        for window in (0, 1, 48, 64, 1024):
            for n in (2, 65, 4096):
                for Hkv in (1, 2, 16):
                    assert chain_pays(3, 16, Hkv, d, window, n, 0, 256) in (True, False)
