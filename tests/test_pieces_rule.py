"""Which layers behind the upload of a batch run in pieces of it (gh_pieces.hip), asked without a device."""
import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D

B, H, W = 8, 224, 224
BATCH = 12 * B * H * W
PLACE = 1 << 28   # of each tensor, by default


def _layers(cmds):
    return _ffi.load().gh_pieces_layers((_ffi.GhCmd * len(cmds))(*cmds), len(cmds))


def _at(i):
    return (i + 1) * PLACE


FILTERS, POOLED = 4 * 16 * 3 * 9, 4 * B * 16 * 112 * 112


def _net(place=None):
    """A convolution and two poolings; `place`: where tensors lie: 0 the batch, 1 the filters, 2 to 4 results, 5 the pinned memory."""
    at = {i: _at(i) for i in range(6)}
    at.update(place or {})
    return [D.cmd_copy(at[0], at[5], BATCH),
            D.cmd_conv2d(at[0], at[1], at[2], B, 3, H, W, 16, 3, 3, (1, 1)),
            D.cmd_maxpool2d(at[2], at[3], B, 16, H, W, 2, 2, (0, 0, 0, 0), (2, 2)),
            D.cmd_maxpool2d(at[3], at[4], B, 16, 112, 112, 2, 2, (0, 0, 0, 0), (2, 2))]


def test_apart():
    cmds = _net()
    assert [_layers(cmds[:n]) for n in range(1, 5)] == [0, 1, 2, 3]
    cmds[0].dim[0] -= 4   # not the batch
    assert _layers(cmds) == 0


# a later layer's result over the filters of the one in front, whole, by its last and by its first bytes, and beside them; its own
@pytest.mark.parametrize("place,layers", [({3: _at(1)}, 1), ({3: _at(1) + FILTERS - 4}, 1), ({3: _at(1) - POOLED + 4}, 1), ({4: _at(1)}, 2), ({2: _at(1)}, 0),
                                          ({3: _at(1) + FILTERS}, 3), ({3: _at(1) - POOLED}, 3)])
def test_a_result_over_filters(place, layers):
    """The layer in front reads its filters again for the next piece, when the first piece's results are there."""
    assert _layers(_net(place)) == layers


@pytest.mark.parametrize("constant", [3, 4, 5, 6])
def test_a_result_over_constants(constant):
    x, w, y, z, bn = (_at(i) for i in range(5))

    def cmds(out):
        conv = D.cmd_conv2d(x, w, y, B, 3, H, W, 16, 3, 3, (1, 1), bn=[bn + 64 * k for k in range(3, 7)])
        return [D.cmd_copy(x, _at(9), BATCH), conv, D.cmd_maxpool2d(y, out, B, 16, H, W, 2, 2, (0, 0, 0, 0), (2, 2))]
    assert _layers(cmds(z)) == 2 and _layers(cmds(bn + 64 * constant + 60)) == 1


# the pooled values read as images of more and of fewer values than were written for one, in a command that is valid by itself
@pytest.mark.parametrize("channels,layers", [(16, 3), (17, 2), (15, 2), (8, 2), (32, 2)])
def test_images_of_another_size(channels, layers):
    cmds = _net()
    cmds[3] = D.cmd_maxpool2d(_at(3), _at(4), B, channels, 112, 112, 2, 2, (0, 0, 0, 0), (2, 2))
    assert _layers(cmds) == layers


# kernels that cut the channels by the number of images: gathering, tiled through LDS, small images
@pytest.mark.parametrize("conv", [D.cmd_conv2d(_at(0), _at(1), _at(2), B, 3, H, W, 64, 16, 16, (0, 0), (16, 16)), D.cmd_conv2d(_at(0), _at(1), _at(2), B, 3, H, W, 16, 5, 5, (2, 2)),
                                  D.cmd_conv2d(_at(0), _at(1), _at(2), B, 588, 16, 16, 16, 3, 3, (1, 1)), D.cmd_conv2d(_at(0), _at(1), _at(2), 96, 64, 14, 14, 64, 3, 3, (1, 1))])
def test_kernels_whose_sums_depend_on_the_number_of_images(conv):
    bytes_ = 4 * conv.dim[0] * conv.dim[1] * conv.dim[2] * conv.dim[3]
    assert bytes_ >= 4000000 and _layers([D.cmd_copy(_at(0), _at(9), bytes_), conv]) == 0
    pool = D.cmd_maxpool2d(_at(0), _at(2), *conv.dim[:4], 2, 2, (0, 0), (2, 2))
    assert _layers([D.cmd_copy(_at(0), _at(9), bytes_), pool]) == 1
