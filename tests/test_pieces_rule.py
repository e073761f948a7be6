"""Which layers behind the upload of a batch run in pieces of it (gh_pieces.hip), asked without a device."""
import numpy as np
import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D
from gorgonia_amd import graph as G

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


def _program(lend, resident=False, more=0):
    """What a compiled machine frees behind each operator: input nodes by name; a convolution, 2 + `more` poolings and a Rectify."""
    g = G.NewGraph()
    x = G.NewTensor(g, np.zeros((B, 3, H, W), np.float32))
    w = G.NewTensor(g, np.zeros((16, 3, 3, 3), np.float32), resident=resident)
    if lend:
        G.LetBorrowed(x)
    nodes = [G.Conv2d(x, w, (3, 3), (1, 1), (1, 1), (1, 1))]
    for _ in range(2 + more):
        nodes.append(G.MaxPool2D(nodes[-1], (2, 2), (0, 0), (2, 2)))
    G.Read(G.Rectify(nodes[-1]))
    m = G.NewTapeMachine(g, compile_only=True)
    lines, behind, names = [l.split("\t")[1].split() for l in m.program().splitlines() if "\t" in l], [], {}
    for l in lines:
        if l[0] == "alloc":
            names[l[3]] = {x.id: "x", w.id: "w"}.get(int(l[2]), int(l[2]) - nodes[0].id)
        if l[0] == "execOp":
            behind.append([])
        if l[0] == "free" and behind:
            behind[-1].append(names[l[3]])
    m.Close()
    return [sorted(map(str, b)) for b in behind[:3 + more]]


def test_a_lent_batch_keeps_what_its_layers_read():
    """Until the last layer that runs in pieces: behind the second pooling here, and of five layers behind the third."""
    assert _program(True) == [[], [], ["0", "1", "w", "x"]]
    assert _program(True, resident=True) == [[], [], ["0", "1", "x"]]
    far = _program(True, more=3)
    kept = next(i for i, b in enumerate(far) if b)
    assert far[kept] == sorted([str(i) for i in range(kept)] + ["w", "x"]) and far[kept + 1:] == [[str(i)] for i in range(kept, 5)]


def test_a_batch_bound_with_let_keeps_nothing():
    """It never runs in pieces: every value goes with its reader."""
    assert _program(False) == [["w", "x"], ["0"], ["1"]]


def test_the_same_answer_when_asked_again(monkeypatch):
    """More shapes than are kept, each asked at different times and with kernels taken out of the choice."""
    def ask(c, f, h, b, pool2):
        y = _at(2)
        cmds = [D.cmd_copy(_at(0), _at(9), 4 * b * c * h * h), D.cmd_conv2d(_at(0), _at(1), y, b, c, h, h, f, 3, 3, (1, 1), pool2=pool2, act="relu")]
        return _layers(cmds)
    shapes = [(c, f, h, -(-4200000 // (4 * c * h * h)) + more, p) for c in (3, 16, 32, 64, 588) for f in (16, 64) for h in (52, 104) for more in (2, 5) for p in (False, True)]
    first = [ask(*s) for s in shapes]
    assert len(shapes) > 64 and set(first) == {0, 1}
    with monkeypatch.context() as p:
        p.setenv("GORGONIA_HIP_CONV_NO_LANES", "1")
        without = [ask(*s) for s in shapes]
    assert without != first
    assert [ask(*s) for s in shapes] == first and [ask(*s) for s in shapes[::-1]] == first[::-1]


def test_the_answer_for_another_alignment():
    """A 1x1 convolution runs on k_conv1x1 where its filters lie at whole lines, else on a kernel that cuts the channels by the images."""
    def ask(w):
        return _layers([D.cmd_copy(_at(0), _at(9), 4 * 8 * 256 * 28 * 28), D.cmd_conv2d(_at(0), w, _at(2), 8, 256, 28, 28, 64, 1, 1)])
    assert [ask(_at(1) + off) for off in (0, 4, 8, 16, 4)] == [1, 0, 0, 1, 0]


@pytest.mark.parametrize("switch,conv", [("POINTWISE", (8, 256, 28, 28, 64, 1, 1)), ("DIRECT", (1024, 2, 32, 32, 16, 3, 3, (1, 1)))])
def test_the_answer_with_a_kernel_taken_out(monkeypatch, switch, conv):
    """The next kernel's cuts the channels by the images; asked before and behind."""
    def ask():
        bytes_ = 4 * conv[0] * conv[1] * conv[2] * conv[3]
        return _layers([D.cmd_copy(_at(0), _at(9), bytes_), D.cmd_conv2d(_at(0), _at(1), _at(2), *conv)])
    assert ask() == 1
    with monkeypatch.context() as p:
        p.setenv("GORGONIA_HIP_CONV_NO_" + switch, "1")
        assert ask() == 0
    assert ask() == 1
