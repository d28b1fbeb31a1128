"""Gated linear attention over blocks of 32 tokens, and over chunks of 16 where values are narrow: lengths around the edges of chunks and
blocks, every width of key and value, several sequences and segments, channels that fade at once beside ones that last."""
import pytest
import torch

from oracle import gitopel as O

pytestmark = pytest.mark.gpu


def portions(lens):
    crow, clen, cu, at = [], [], [0], 0
    for n in lens:
        crow += list(range(at, at + n, 16))
        clen += [min(16, n - c) for c in range(0, n, 16)]
        cu.append(len(crow))
        at += n
    return [torch.tensor(x, dtype=torch.int32, device="cuda") for x in (crow, clen, cu)]


def run(H, dk, dv, rank, lens, start, tau, seed, lost=None, scale=1.0, known=True):
    from tinyllmforge_amd import ops as P
    g, dt, eps = torch.Generator().manual_seed(seed), torch.bfloat16, 1e-5
    proj = [torch.randn(n, 2 * H * (dk + dv) + rank, generator=g).to(dt) for n in lens]
    for p in proj:
        p[:, H * dk:2 * H * dk] *= scale
        p[:, :H * dk] /= scale
    a2, a2b, nw = torch.randn(H * dk, rank, generator=g).to(dt), 2 + torch.randn(H * dk, generator=g).to(dt), torch.randn(dv, generator=g).to(dt)
    a2[::7] *= 4                                             # some channels fade much faster than others
    if lost is not None:
        proj[lost][:] = float("nan")
    first = [torch.randn(H, dk, dv, generator=g) for _ in lens]
    state = torch.stack([torch.full((H, dk, dv), 5.0)] + first).cuda()
    out = torch.full((sum(lens), H * dv), 7.0, dtype=dt, device="cuda")
    t = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    P.gla_portions(torch.cat(proj).cuda(), a2.cuda(), a2b.cuda(), nw.cuda(), state, t([i + 1 for i in range(len(lens))]), t(start), *portions(lens), 0, len(lens),
                   tau, eps, out, max(lens) if known else 0)
    assert (state[0] == 5.0).all()
    at, errs = 0, []
    for i, n in enumerate(lens):
        if i != lost:
            p = proj[i].double()
            q, k, v, gt, r = p.split([H * dk, H * dk, H * dv, H * dv, rank], dim=1)
            la = -torch.nn.functional.softplus(-(r @ a2.double().T + a2b.double())).view(-1, H, dk) / tau
            o, s = O.gla_recurrence(q.view(-1, H, dk) * dk ** -0.5, k.view(-1, H, dk), v.view(-1, H, dv), la, first[i].double() if start[i] else None)
            want = (O.unit_rms(o, eps) * nw.double()).reshape(-1, H * dv) * O.silu(gt)
            err = lambda a, b: ((a.double().cpu() - b).norm() / b.norm()).item()
            errs.append((n, err(out[at:at + n], want), err(state[i + 1], s)))
        at += n
    return errs


# The output is rounded to bfloat16, by at most 2^-8 of each value.  Products are exact to 2^-24 and sums of 32 tokens' logarithms
# towards the block's end (below 16 where a power still counts, to 2^-20 in the exponent) are in single precision.
OUT, STATE = 2 ** -8, 2 ** -20


@pytest.mark.parametrize("dk,dv", [(32, 32), (32, 64), (32, 256), (64, 96), (128, 64), (128, 96), (128, 256)])
@pytest.mark.parametrize("tau", [16.0, 0.25])
def test_lengths_around_chunks_and_blocks(dk, dv, tau):
    lens = [1, 15, 16, 17, 31, 32, 33, 47, 49, 63, 64, 65]
    for n, out, state in run(2, dk, dv, 16, lens, [5 * (i % 2) for i in range(len(lens))], tau, dk + dv):
        assert out < OUT and state < STATE, (n, out, state)


@pytest.mark.parametrize("dk,dv,rank,lens", [(128, 64, 8, [2100]), (128, 96, 8, [2100]), (64, 64, 64, [1500, 700, 33]), (32, 64, 24, [513, 2000])])
def test_segments_of_whole_blocks(dk, dv, rank, lens):
    for n, out, state in run(1, dk, dv, rank, lens, [0] + [3] * (len(lens) - 1), 8.0, dk):
        assert out < OUT and state < STATE, (n, out, state)


def test_keys_that_leave_no_room_for_growing_powers():
    for n, out, state in run(1, 64, 64, 16, [70], [0], 8.0, 3, scale=1e25):
        assert out < OUT and state < STATE, (n, out, state)


@pytest.mark.parametrize("dv", [64, 128])
@pytest.mark.parametrize("lost", [0, 1, 2])
def test_rows_of_another_sequence_are_not_touched(lost, dv):
    for n, out, state in run(2, 128, dv, 16, [17, 40, 50], [0, 5, 5], 16.0, lost, lost=lost):
        assert out < OUT and state < STATE, (n, out, state)


@pytest.mark.parametrize("dk,dv", [(32, 64), (64, 128), (128, 32), (128, 256)])
@pytest.mark.parametrize("token", [16, 20, 31, 50])
def test_a_value_without_a_number_reaches_no_earlier_chunk(dk, dv, token):
    """Sixteen tokens are a chunk; an earlier token meets values behind it as zeros times them."""
    from tinyllmforge_amd import ops as P
    H, rank, n = 2, 16, 60
    g, dt = torch.Generator().manual_seed(token), torch.bfloat16
    proj = torch.randn(n, 2 * H * (dk + dv) + rank, generator=g).to(dt).cuda()
    a2, a2b, nw = (torch.randn(s, generator=g).to(dt).cuda() for s in ((H * dk, rank), (H * dk,), (dv,)))
    t = lambda *x: torch.tensor(x, dtype=torch.int32, device="cuda")
    def run():
        out = torch.full((n, H * dv), 7.0, dtype=dt, device="cuda")
        P.gla_portions(proj, a2, a2b, nw, torch.zeros(1, H, dk, dv, device="cuda"), t(0), t(0), *portions([n]), 0, 1, 8.0, 1e-5, out)
        return out
    want = run()
    for value in (torch.nan, torch.inf):
        proj[token, 2 * H * dk:2 * H * dk + H * dv] = value
        got, first = run(), token // 16 * 16
        assert torch.equal(got[:first], want[:first]) and not got[token:].isfinite().any()


@pytest.mark.parametrize("dk,dv", [(48, 40), (100, 32), (256, 64)])
@pytest.mark.parametrize("tau", [16.0, 0.25])
def test_other_sizes_in_chunks_of_16_tokens(dk, dv, tau):
    lens = [1, 15, 16, 17, 31, 33, 200]
    for n, out, state in run(2, dk, dv, 16, lens, [5 * (i % 2) for i in range(len(lens))], tau, dk + dv):
        assert out < OUT and state < STATE, (n, out, state)


@pytest.mark.parametrize("H,dk,dv,lens,kernels", [
    (16, 128, 256, [64], 2), (16, 128, 256, [65], 3), (16, 128, 256, [400], 3), (16, 128, 256, [200] * 5, 2), (16, 128, 256, [600], 4),
    (8, 64, 128, [200], 2), (8, 64, 128, [224, 209], 3), (8, 64, 128, [240] * 12, 2), (16, 128, 128, [500] * 8, 3)])
def test_short_portions_keep_the_chunks(H, dk, dv, lens, kernels):
    """Two kernels over blocks of 32 tokens, two more where there are segments; three over chunks of 16."""
    from tinyllmforge_amd import _lib
    count = _lib.load().tlf_kernel_launches
    before = count()
    for n, out, state in run(H, dk, dv, 16, lens, [5] * len(lens), 8.0, dk):
        assert out < OUT and state < STATE, (n, out, state)
    assert count() - before == kernels


@pytest.mark.parametrize("lens,start", [([1500, 33, 1700, 2, 1024, 32], [0, 5, 7, 0, 64, 0]), ([2047], [3]), ([512, 512, 512, 512], [0, 1, 0, 1]),
                                        ([17, 3000, 31, 40], [1, 1, 0, 9]), ([700, 1, 900], [1, 1, 1])], ids=str)
@pytest.mark.parametrize("H,dk,dv", [(2, 128, 256), (3, 64, 96)])
def test_stretches_over_sequences(H, dk, dv, lens, start):
    """Stretches that begin and end anywhere: within a sequence, at its ends, several sequences in one, one sequence in many."""
    from tinyllmforge_amd import _lib
    count = _lib.load().tlf_kernel_launches
    before = count()
    for n, out, state in run(H, dk, dv, 16, lens, start, 16.0, sum(lens)):
        assert out < OUT and state < STATE, (n, out, state)
    assert count() - before == 4                             # blocks, what stretches add, the states they start from, the scan


@pytest.mark.parametrize("dk", [64, 128])
@pytest.mark.parametrize("dv", [160, 192, 224, 256])           # five to eight waves: the fifth and later finish a block behind their products
@pytest.mark.parametrize("lens,start", [([1], [3]), ([33, 95, 64], [0, 1, 1]), ([1500, 40], [5, 0])])
def test_waves_that_share_a_simd(dk, dv, lens, start):
    for n, out, state in run(2, dk, dv, 8, lens, start, 16.0, seed=dv + len(lens)):
        assert out < OUT and state < STATE, (n, out, state)


@pytest.mark.parametrize("seqs", [16, 17, 32, 33, 63, 64, 65])
def test_stretches_over_many_sequences(seqs):
    """A lane for each sequence, up to all 64 of them; one more makes two groups."""
    from tinyllmforge_amd import _lib
    count = _lib.load().tlf_kernel_launches
    before, lens = count(), [600 + 37 * (5 * i % 7) - 90 * (i % 3) for i in range(seqs)]
    lens[40 % seqs] += 4000 * (seqs > 64)                    # groups are cut for a long one only
    for n, out, state in run(1, 32, 64, 16, lens, [i % 2 for i in range(seqs)], 16.0, seqs):
        assert out < OUT and state < STATE, (n, out, state)
    assert count() - before == (4 if seqs <= 64 else 7)


# 64 heads of 32 x 64: 512 workgroups fill the chip, 8 stretches of 64 heads; 7 heads: 73 stretches, in two groups of up to 64 sequences
@pytest.mark.parametrize("H,lens,known,kernels", [(64, [2500] + [130] * 5, True, 4), (64, [130] * 5 + [2500], True, 4), (64, [520] * 6, True, 2), (64, [520] * 6, False, 4),
                                                  (7, [470] * 32 + [4000] + [470] * 32, True, 7), (7, [512] * 65, True, 2)],
                         ids=["long first", "long last", "alike", "not known", "more than 64", "more than 64 alike"])
def test_one_long_sequence_among_short_ones(H, lens, known, kernels):
    """Hardly more stretches than sequences: they are cut where one is much longer than an even share."""
    from tinyllmforge_amd import _lib
    count = _lib.load().tlf_kernel_launches
    before = count()
    for n, out, state in run(H, 32, 64, 16, lens, [i % 3 for i in range(len(lens))], 16.0, H, known=known):
        assert out < OUT and state < STATE, (n, out, state)
    assert count() - before == kernels


@pytest.mark.parametrize("rank", [1, 5, 8, 17, 24, 40, 63])
@pytest.mark.parametrize("dk,dv", [(32, 64), (128, 96)])
def test_ranks_of_the_decays_projection(dk, dv, rank):
    """As with a rank of 64 whose other columns are zeros; what lies behind a row's own columns is not read."""
    from tinyllmforge_amd import ops as P
    H, lens = 2, [33, 100, 520]
    g, dt, n = torch.Generator().manual_seed(rank), torch.bfloat16, sum(lens)
    head = torch.randn(n, 2 * H * (dk + dv), generator=g).to(dt)
    r, a2 = torch.randn(n, rank, generator=g).to(dt), torch.randn(H * dk, rank, generator=g).to(dt)
    a2b, nw = 1 + torch.randn(H * dk, generator=g).to(dt), torch.randn(dv, generator=g).to(dt)
    t = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    zeros = torch.nn.functional.pad
    res = []
    for rows, weights, behind in ((r, a2, float("nan")), (zeros(r, (0, 64 - rank)), zeros(a2, (0, 64 - rank)), 0.0)):
        proj = torch.full((n, -(-(head.shape[1] + rows.shape[1]) // 8) * 8 + 8), behind, dtype=dt)
        proj[:, :head.shape[1]], proj[:, head.shape[1]:head.shape[1] + rows.shape[1]] = head, rows
        state, out = torch.zeros(3, H, dk, dv, device="cuda"), torch.zeros(n, H * dv, dtype=dt, device="cuda")
        P.gla_portions(proj.cuda(), weights.cuda(), a2b.cuda(), nw.cuda(), state, t([0, 1, 2]), t([0, 0, 0]), *portions(lens), 0, 3, 8.0, 1e-5, out, 520)
        res.append((out, state))
    assert all(x.isfinite().all() and torch.equal(x, y) for x, y in zip(*res))
