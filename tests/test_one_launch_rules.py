"""When a decoding step or an encoder runs in one launch, and what it refuses: host code
alone where nothing says gpu."""

import ctypes

import pytest

from fei_amd import ops
from fei_amd.ops.layers import _EncoderShape, _OneShape


def room(kind, blocks):
    lib = ops.require_lib()
    if kind == "step":
        return lib.fei_decode_one_room(ctypes.byref(_OneShape(
            2, 2048, 8192, 32, 8, 64, 320, 4000, 0, blocks, 1e-5, 0.125)))
    return lib.fei_encoder_one_room(ctypes.byref(_EncoderShape(
        2, 1, 24, 12, 768, 3072, blocks, 1e-5, 0.125)))


@pytest.mark.parametrize("kind", ["step", "encoder"])
def test_blocks_of_a_launch(kind):
    """More than there are items would have items of their own past every end."""
    want = room(kind, 256)
    assert want > 0
    for blocks in (1, 2, 255):
        assert room(kind, blocks) == want
    for blocks in (-1, 0, 257, 512):
        assert room(kind, blocks) == 0
