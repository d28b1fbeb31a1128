"""State-space portions with the heads of a group in one workgroup: lengths around the edges of chunks, workgroups that are not full, every
state size, heads whose decay leaves the common scale, segments."""
import pytest
import torch

from tests.test_gpu_tibenex import rel, run_ssd, ssd_case

pytestmark = pytest.mark.gpu
BF = torch.bfloat16
# x, B and C are rounded to bfloat16 before the sums and y * silu(z) after them: four relative errors of at most 2^-9 on average over
# a product, three of them of one term's factors.
TOL = 4 * 2 ** -9 * 0.77


def copies(sizes, seqs):
    """How often so many short sequences make 256 workgroups of 8 x 32 columns."""
    H, Pv, N, G, taps = sizes
    return -(-256 // (seqs * G * -(-(H // G * Pv // 32) // 8)))


@pytest.mark.parametrize("sizes", [(24, 64, 128, 8, 4), (32, 32, 64, 8, 3), (64, 96, 32, 16, 4), (32, 64, 128, 4, 4), (40, 64, 64, 4, 2)])
@pytest.mark.parametrize("decay,step", [(0.0, -1.5), (-4.0, -3.0), (3.0, 3.0), (2.0, 0.0)])
def test_lengths_around_chunks(sizes, decay, step):
    """Whole prompts, and a second portion that starts from the first one's state; the last two decays leave 2^63 within a chunk for
    every head, and for some."""
    lens = [2, 63, 64, 65, 127, 129]
    proj, w, want = ssd_case(sizes, lens, BF, sum(sizes), decay, step)
    times = copies(sizes, len(lens))
    for steps in ([lens], [[0, 50, 60, 2, 64, 65], [2, 13, 4, 63, 63, 64]]):
        got = run_ssd(sizes, proj * times, w, [x * times for x in steps], BF, list(range(1, 6 * times + 1)))
        for s in list(range(6)) + list(range(6 * times - 6, 6 * times)):
            assert rel(got[s], want[s % 6]) < TOL, (steps[0][s % 6], s, rel(got[s], want[s % 6]))


@pytest.mark.parametrize("sizes,lens", [((64, 32, 128, 8, 4), [1500, 300]), ((32, 64, 32, 8, 4), [4111]), ((64, 64, 64, 8, 4), [600, 2, 1000])])
def test_segments(sizes, lens):
    """Sequences cut into segments, of which short ones leave some empty; late rows still see the first through a slow decay."""
    proj, w, want = ssd_case(sizes, lens, BF, 5, decay=-5.0, step=-3.0)
    for first in (0, 70):
        steps = ([[min(first, n - 2) for n in lens]] if first else []) + [[n - (min(first, n - 2) if first else 0) for n in lens]]
        got = run_ssd(sizes, proj, w, steps, BF, list(range(1, len(lens) + 1)))
        for s in range(len(lens)):
            assert rel(got[s], want[s]) < TOL, (first, s)
            assert rel(got[s][-50:], want[s][-50:]) < 8e-3, (first, s)


@pytest.mark.parametrize("sizes,lens,lost", [((64, 64, 64, 8, 4), [670] * 8, True), ((64, 64, 128, 8, 4), [1170, 1071, 970, 1170], False),
                                             ((32, 64, 32, 8, 4), [770, 72, 700, 770], False)])
def test_beginnings_that_are_gone_through_once(sizes, lens, lost):
    """The first pass goes through a chunk or two of each long sequence for good, from nothing and from a state of its own; of a short one
    through none, which hands its state on.  A sequence without a place for its state takes none along."""
    proj, w, want = ssd_case(sizes, lens, BF, 9, decay=-5.0, step=-3.0)
    slots = list(range(1, len(lens) + 1))
    if lost:
        slots[1] = -1
    for steps in ([lens], [[70] * len(lens), [n - 70 for n in lens]]):
        got = run_ssd(sizes, proj, w, steps, BF, slots)
        for s in range(len(lens)):
            if slots[s] > 0 or len(steps) == 1:
                assert rel(got[s], want[s]) < TOL and rel(got[s][-50:], want[s][-50:]) < 8e-3, s


@pytest.mark.parametrize("sizes", [(16, 64, 64, 8, 4), (24, 64, 128, 8, 4), (56, 32, 32, 8, 4)])
def test_first_passes_without_beginnings(sizes):
    """Sequences enough for half the chip: the first pass only gathers, in less LDS, and hands the states on that are there."""
    lens, times = [1160, 300, 700], 9
    proj, w, want = ssd_case(sizes, lens, BF, 11, decay=-5.0, step=-3.0)
    slots = list(range(1, 3 * times + 1))
    slots[4] = -1
    for steps in ([lens], [[70, 2, 64], [1090, 298, 636]], [[8, 140, 1], [1152, 160, 699]]):
        got = run_ssd(sizes, proj * times, w, [x * times for x in steps], BF, slots)
        for s in range(3 * times):
            if slots[s] > 0 or len(steps) == 1:
                assert rel(got[s], want[s % 3]) < TOL and rel(got[s][-50:], want[s % 3][-50:]) < 8e-3, s


@pytest.mark.parametrize("sizes", [(24, 64, 128, 8, 4), (32, 32, 64, 8, 3), (64, 96, 32, 16, 4)])
def test_portions_behind_single_tokens(sizes):
    """A step's single tokens come first: portions begin at rows and sequences of their own, in the inputs and behind the convolution.
    The last step's tokens see the states that the portions left (a row alone: errors that do not average out)."""
    steps = [[50, 1, 2, 64, 1, 65], [13, 1, 63, 1, 70, 1], [1, 1, 1, 1, 1, 1]]
    lens = [sum(x) for x in zip(*steps)]
    proj, w, want = ssd_case(sizes, lens, BF, sum(sizes), 0.0, -1.5)
    times = copies(sizes, 3)
    got = run_ssd(sizes, proj * times, w, [x * times for x in steps], BF, list(range(1, 6 * times + 1)))
    for s in list(range(6)) + list(range(6 * times - 6, 6 * times)):
        assert rel(got[s], want[s % 6]) < TOL and rel(got[s][-1], want[s % 6][-1]) < 2 * TOL, (s, rel(got[s], want[s % 6]))


@pytest.mark.parametrize("sizes", [(64, 32, 128, 8, 4), (64, 64, 64, 8, 4)])
def test_segments_behind_single_tokens(sizes):
    steps = [[700, 1, 100, 1], [800, 1, 200, 1], [1, 1, 1, 1]]
    lens = [sum(x) for x in zip(*steps)]
    proj, w, want = ssd_case(sizes, lens, BF, 7, decay=-5.0, step=-3.0)
    got = run_ssd(sizes, proj, w, steps, BF, [3, 0, 2, 1])
    for s in range(4):
        assert rel(got[s], want[s]) < TOL and rel(got[s][-1], want[s][-1]) < 2 * TOL, s


@pytest.mark.parametrize("state_dim", [32, 64, 128])
def test_the_state_is_summed_in_single_precision(state_dim):
    """Sums of three tokens, whose factors no rounding to bfloat16 touches: x, B and C pass the convolution and SiLU as they are, and
    softplus leaves the step sizes."""
    from tinyllmforge_amd import ops as P
    H, Pv, G, seqs, n = 24, 64, 8, 64, 3
    inner, chan = H * Pv, H * Pv + 2 * G * state_dim
    g = torch.Generator().manual_seed(state_dim)
    between = lambda lo, hi, *s: (lo + (hi - lo) * torch.rand(*s, generator=g)).to(BF)
    proj = torch.cat([torch.zeros(seqs * n, inner), between(32, 64, seqs * n, chan), between(20, 30, seqs * n, H)], dim=1).to(BF)
    conv, a_log = torch.zeros(4, chan, dtype=BF), between(-6, -4, H)
    conv[-1] = 1
    w = P.SsdWeights(conv.cuda(), torch.zeros(chan, dtype=BF).cuda(), torch.zeros(H, dtype=BF).cuda(), a_log.cuda(), torch.ones(H, dtype=BF).cuda())
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    state, ring = torch.full((seqs, H, state_dim, Pv), 5.0, device="cuda"), torch.zeros(seqs, 4, chan, dtype=BF, device="cuda")
    out = torch.empty(seqs * n, inner, dtype=BF, device="cuda")
    P.ssd_portions(proj.cuda(), w, ring, state, i32(range(seqs)), torch.arange(n).repeat(seqs).cuda(), i32([s for s in range(seqs) for _ in range(n)]),
                   i32(range(0, seqs * n + 1, n)), i32([0] * seqs), 0, seqs, 0, n, G, out)
    x, B, _, dt = proj[:, inner:].double().view(seqs, n, -1).split([inner, G * state_dim, G * state_dim, H], dim=2)
    x, B = x.view(seqs, n, H, Pv), B.reshape(seqs, n, G, state_dim).repeat_interleave(H // G, 2)
    want = torch.zeros(seqs, H, state_dim, Pv, dtype=torch.float64)
    for t in range(n):
        want = want * torch.exp(-torch.exp(a_log.double()) * dt[:, t])[..., None, None] + (dt[:, t, :, None] * B[:, t])[..., None] * x[:, t, :, None]
    # a factor's roundings (an exponential, two products) and those of three sums, at most 2^-23 each and half of that on average; with
    # pairs of bfloat16, 2^-17 at most for each token, the sums were 2^-20 off and more
    assert rel(state, want) < 2 ** -21
