"""The recurrences with a matrix state over prompts that are cut into segments: a prompt taken whole and in portions that
are too short to be cut leave the same states and the same outputs, for every mixer on that recurrence."""

import pytest
import torch

from test_mogisun_mechanisms import context, lowered, rnd
from simple_inference_amd.parts.context import LayerCache

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def run(op, k, rows, H, D, Dv, lengths, portion):
    """Outputs and states of the sequences, every step bringing each of them up to ``portion`` more tokens, and whether any
    step was cut: whether it wrote into its workspace behind the decays and the raw outputs."""
    g = torch.Generator().manual_seed(5)
    f32 = lambda t: t.float().to(DEV)
    bf16 = lambda t: t.to(torch.bfloat16).to(DEV)
    state = torch.zeros(len(lengths) + 2, H * D * Dv, device=DEV)
    state[0].fill_(0.25)                     # the first sequence goes on from a state
    norm, bias, lower = f32(1 + rnd(g, Dv, std=0.2)), f32(rnd(g, H * D)), f32(torch.rand(H * D, generator=g) * 0.9)
    per_head, decays = f32(1 + rnd(g, H * Dv, std=0.2)), f32(0.9 + 0.0999 * torch.rand(H, generator=g))
    a2, out = bf16(rnd(g, H * D, 32, std=0.3)), torch.empty(sum(lengths), H * Dv)
    offsets, at = [sum(lengths[:s]) for s in range(len(lengths))], [0] * len(lengths)
    was_cut = False
    while any(a < n for a, n in zip(at, lengths)):
        who = [s for s, n in enumerate(lengths) if at[s] < n]
        lens = [min(portion, lengths[s] - at[s]) for s in who]
        idx = torch.cat([torch.arange(offsets[s] + at[s], offsets[s] + at[s] + n) for s, n in zip(who, lens)])
        ctx, x = context(DEV, lens, who), rows[idx.to(DEV)].contiguous()
        qk, v = H * D, H * Dv
        space = ctx.recurrent_workspace = torch.full((sum(lens) * (2 * qk + v) + 2 * (sum(lens) // 64 + 1) * qk * Dv + 4,), float("nan"), device=DEV)
        if op == "gla":
            y = k.gla_recurrent(x, (0, qk, 2 * qk, 2 * qk + v, 2 * qk + 2 * v), a2, bias, norm, H, D, Dv, 8.0, D ** -0.5, 1e-5, ctx,
                                LayerCache(state=state.view(-1, H, D, Dv)))
        elif op == "hgrn":
            y = k.hgrn2_scan(x[:, :2 * qk + v].contiguous(), bias, lower, norm, H, D, Dv, 1e-5, ctx, state.view(-1, H, D, Dv))
        elif op == "ssd":        # one group: keys and queries are shared by the heads
            proj = x[:, :v + H].contiguous()
            y = k.ssd_scan(proj, x[:, v + H:2 * v + H + 2 * D].contiguous(), f32(decays), f32(-decays), f32(decays), per_head, H, Dv, D,
                           1, 1, 1e-5, ctx, state)
        elif op == "decay":
            y = k.decay_attention(x[:, :2 * qk + 2 * v].contiguous(), decays, per_head, H, D, Dv, 1e-5, ctx, state.view(-1, H, D, Dv))
        else:
            rkvg = torch.stack([x[:, i * qk:(i + 1) * qk] for i in range(4)]).contiguous()
            y = k.bonus_recurrence(rkvg, x[:, -32:].contiguous(), a2, bias - 2.0, bias, per_head, H, D, 1e-5, ctx, state)
        out[idx] = y.float().cpu()
        assert ctx.recurrent_workspace is space
        was_cut |= not space[sum(lens) * ((2 if op in ("hgrn", "ssd") else 1) * qk + v) + (-sum(lens) * qk) % 4:].isnan().all()
        for s, n in zip(who, lens):
            at[s] += n
    return out, state, was_cut


def projected(g, n, H, D, Dv):
    """Rows wide enough for every mixer's columns, a multiple of eight."""
    width = 2 * H * D + 2 * H * Dv + 2 * D + H + 32
    return lowered(rnd(g, n, width + -width % 8), torch.bfloat16, DEV)[0]


# the shortest prompt that is cut and the one just beside it, remainders of a segment from one token on, one token beside
# them; states of more than 128 rows; enough heads for the long segments; sequences enough for the sparse places of
# segments; runs that are walked whole with four columns a lane group; tokens enough for decays on the matrix cores (its
# portions are below); value widths that the cut does not take
@pytest.mark.parametrize("op", ["gla", "hgrn", "ssd", "decay", "bonus"])
@pytest.mark.parametrize("H,D,Dv,lengths,cut", [
    (2, 128, 128, [300, 1, 129, 64, 127], True), (2, 128, 128, [177], True), (2, 128, 128, [176], False),
    (3, 40, 24, [128, 257], True), (1, 200, 104, [191, 130], True), (1, 200, 104, [128], True), (2, 64, 30, [300, 3], False),
    (80, 16, 16, [1300, 128, 2, 385], True), (2, 64, 64, [200, 1, 1, 1, 1, 1, 1, 1, 65], True),
    (8, 128, 128, [130] * 15 + [140], False), (12, 256, 256, [130] * 3, False), (24, 128, 128, [1100], True)])
def test_a_prompt_cut_into_segments_is_the_prompt_walked_along(op, H, D, Dv, lengths, cut):
    """States are sums in float whose order differs by a product of decays taken first (relative 2^-23 a token); outputs
    are rounded to bfloat16 once, so they are equal or neighbours (2^-7 relative)."""
    from simple_inference_amd.kernels import HipKernels

    if op == "bonus":        # square matrices: never a width that the cut does not take
        cut, Dv = cut or Dv % 4 != 0, D
    k = HipKernels()
    g = torch.Generator().manual_seed(H * D)
    rows = projected(g, sum(lengths), H, D, Dv)
    whole, state, was_cut = run(op, k, rows, H, D, Dv, lengths, 10 ** 6)
    portions, want, portions_were_cut = run(op, k, rows, H, D, Dv, lengths, 100)
    assert was_cut == cut and not portions_were_cut
    assert float((state - want).abs().max()) <= 2e-5 * float(want.abs().max())
    assert bool(((whole - portions).abs() <= 2.0 ** -7 * portions.abs() + 1e-3 * float(portions.std())).all()), float((whole - portions).abs().max())
    assert float(state[len(lengths):].abs().max()) == 0.0        # nobody else's slot was touched


@pytest.mark.parametrize("decay", ["usual", "strong", "mixed", "above", "around"])
@pytest.mark.parametrize("H,D,Dv,lengths", [
    (2, 64, 64, [32, 1, 15, 16, 17]), (3, 128, 128, [33, 47, 2]), (2, 80, 192, [100, 31, 1]), (1, 112, 80, [48] * 5), (2, 64, 144, [200, 3]),
    (2, 128, 64, [513]), (1, 128, 128, [177, 300]), (1, 64, 272, [65, 50]), (2, 64, 128, [300, 17]),
    (2, 64, 64, [48, 1, 15, 16, 17]), (3, 128, 128, [49, 63, 2])])
def test_runs_by_blocks_against_64_bits(H, D, Dv, lengths, decay):
    """Whole and cut runs, last blocks of one to 16 tokens, widths that leave waves or channels idle; decays as trained, decays that
    leave nothing within a block (which go pair by pair), and those in some channels only.  Decays that leave a little more than 2^-40 of a
    block (the largest k / P there is), or about that, go one way and the other.  A state's error is that of its decays
    (four units in the last place a token) and of some 100 sums, of what the same recurrence gives with absolute values."""
    from simple_inference_amd.kernels import HipKernels

    k, rank, tau, n = HipKernels(), 32, 16.0, sum(lengths)
    g = torch.Generator().manual_seed(D + Dv)
    cols = (0, H * D, 2 * H * D, 2 * H * D + H * Dv, 2 * H * (D + Dv))
    rows = rnd(g, n, cols[4] + rank).to(torch.bfloat16).to(DEV)
    a2, bias = rnd(g, H * D, rank, std=0.1).to(torch.bfloat16).to(DEV), rnd(g, H * D, std=0.1).to(DEV)
    if decay in ("above", "around"):      # sixteen sixteenths of log sigmoid: 2^-39 and 2^-40
        bias = bias * 0.3 - (39 if decay == "above" else 40) * 0.6931
    elif decay != "usual":
        bias -= 2000.0
    if decay == "mixed":
        bias.view(H, D)[:, :D // 2] += 2000.0
    norm = (1 + rnd(g, Dv, std=0.2)).float().to(DEV)
    state = rnd(g, len(lengths), H, D, Dv).float().to(DEV)
    want, size = state.double(), state.double().abs()
    x = rows.double()
    q, key = (x[:, cols[i]:cols[i] + H * D].view(n, H, D, 1) for i in (0, 1))
    v, gate = (x[:, cols[i]:cols[i] + H * Dv].view(n, H, 1, Dv) for i in (2, 3))
    alpha = torch.exp(torch.nn.functional.logsigmoid(x[:, cols[4]:] @ a2.double().T + bias.double()) / tau).view(n, H, D, 1)
    o, t = torch.empty(n, H, Dv, dtype=torch.float64, device=DEV), 0
    for s, length in enumerate(lengths):
        for _ in range(length):
            want[s] = alpha[t] * want[s] + key[t] * v[t]
            size[s] = alpha[t] * size[s] + (key[t] * v[t]).abs()
            o[t] = (want[s] * q[t]).sum(1) * D ** -0.5
            t += 1
    y = k.gla_recurrent(rows, cols, a2, bias.float(), norm, H, D, Dv, tau, D ** -0.5, 1e-5, context(DEV, lengths, list(range(len(lengths)))),
                        LayerCache(state=state)).double().view(n, H, Dv)
    ref = o * torch.rsqrt((o * o).mean(-1, keepdim=True) + 1e-5) * norm.double() * torch.nn.functional.silu(gate.squeeze(2))
    assert bool(((state.double() - want).abs() <= (4 * max(lengths) + 100) * 2.0 ** -24 * size + 1e-30).all())
    assert bool(((y - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-4 * ref.std()).all()), float((y - ref).abs().max())


@pytest.mark.parametrize("H,D,Dv,lengths", [(2, 64, 64, [50, 16]), (1, 128, 128, [300])])
def test_small_keys_keep_their_bits_in_runs_by_blocks(H, D, Dv, lengths):
    """Keys around 2^-122, whose last bits times a decay lie below what bfloat16 numbers hold: a state's error is as for others (four units
    in the last place a token for the decays, some 100 sums)."""
    from simple_inference_amd.kernels import HipKernels

    k, n, qk, v = HipKernels(), sum(lengths), H * D, H * Dv
    g = torch.Generator().manual_seed(D)
    cols = (0, qk, 2 * qk, 2 * qk + v, 2 * qk + 2 * v)
    rows = rnd(g, n, cols[4] + 32)
    rows[:, qk:2 * qk] *= 2.0 ** -122
    rows = rows.to(torch.bfloat16).to(DEV)
    a2, bias = rnd(g, qk, 32, std=0.1).to(torch.bfloat16).to(DEV), rnd(g, qk, std=0.1).float().to(DEV)
    state = torch.zeros(len(lengths), H, D, Dv, device=DEV)
    want, size, x, t = state.double(), state.double(), rows.double(), 0
    alpha = torch.exp(torch.nn.functional.logsigmoid(x[:, cols[4]:] @ a2.double().T + bias.double()) / 4).view(n, H, D, 1)
    for s, length in enumerate(lengths):
        for _ in range(length):
            added = x[t, qk:2 * qk].view(H, D, 1) * x[t, 2 * qk:cols[3]].view(H, 1, Dv)
            want[s], size[s] = alpha[t] * want[s] + added, alpha[t] * size[s] + added.abs()
            t += 1
    k.gla_recurrent(rows, cols, a2, bias, torch.ones(Dv, device=DEV), H, D, Dv, 4.0, D ** -0.5, 1e-5,
                    context(DEV, lengths, list(range(len(lengths)))), LayerCache(state=state))
    assert bool(((state.double() - want).abs() <= (4 * max(lengths) + 100) * 2.0 ** -24 * size + n * 2.0 ** -149).all()), float(((state.double() - want).abs() / size).max())


@pytest.mark.parametrize("op", ["gla", "hgrn", "ssd", "decay", "bonus"])
@pytest.mark.parametrize("H,D,Dv,lengths", [(2, 128, 128, [70, 41]), (2, 64, 64, [300, 64]), (1, 128, 64, [200, 100])])
def test_numbers_without_bounds_reach_no_earlier_token(op, H, D, Dv, lengths):
    """Infinities, NaN and numbers whose products leave the range of floats, in the columns of queries, keys and values: blocks of tokens
    give what the tokens one after the other give, NaN in the same places, and finite results in front of them.  (At 2^127 whether a sum of
    128 such products overflows on its way is a matter of its order; 2^110 leaves it 2^17.  An infinite state is NaN behind a whole segment whose decays' product is zero.)"""
    from simple_inference_amd.kernels import HipKernels

    if op == "bonus":
        Dv = D
    k, n = HipKernels(), sum(lengths)
    clean = projected(torch.Generator().manual_seed(D), n, H, D, Dv)
    for at, column in ((21, 3), (37, H * D + 5), (46, 2 * H * D + 9), (lengths[0] + 20, H * D + 8)):
        for value in (float("inf"), float("-inf"), float("nan"), 2.0 ** 100, -2.0 ** 110):
            rows = clean.clone()
            rows[at, column] = value
            whole, state, _ = run(op, k, rows, H, D, Dv, lengths, 10 ** 6)
            tokens, want, _ = run(op, k, rows, H, D, Dv, lengths, 16)
            first = 0 if at < lengths[0] else lengths[0]
            assert bool(whole[first:at].isfinite().all()), (at, column, value)
            assert torch.equal(whole.isnan(), tokens.isnan()) and torch.equal(state.isfinite(), want.isfinite()), (at, column, value)
            spread = 1e-3 * float(tokens[tokens.isfinite()].std())
            assert bool(((whole - tokens).abs() <= 2.0 ** -7 * tokens.abs() + spread)[tokens.isfinite()].all()), (at, column, value)
            same = want.isfinite()
            assert float((state - want)[same].abs().max()) <= 2e-5 * float(want[same].abs().max()), (at, column, value)


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("H,Dv,n", [(1, 8, 3), (3, 24, 33), (5, 64, 51), (2, 136, 40), (3, 256, 7), (2, 512, 129), (3, 20, 33), (20, 20, 1010)])
def test_norm_and_gate_behind_a_prompt_s_recurrence(H, Dv, n, shift):
    """Groups of one to 64 lanes a (token, head), lanes without elements, a last workgroup in part, and rows that do not begin at 16
    bytes or divide into eights (the general form: a (token, head) a wave, and four where there are many).  With decays and keys that leave the outputs q k v of one channel, each is known to a few
    roundings of float; the result is rounded once to bfloat16 (2^-9)."""
    from simple_inference_amd.kernels import HipKernels

    k, D, rank, eps = HipKernels(), 16, 8, 1e-5
    g = torch.Generator().manual_seed(Dv + shift)
    cols = (0, H * D, 2 * H * D, 2 * H * D + H * Dv + shift, 2 * H * (D + Dv) + 8)
    rows = rnd(g, n, cols[4] + rank).to(torch.bfloat16)
    a2, bias = torch.zeros(H * D, rank, dtype=torch.bfloat16), torch.full((H * D,), -1e6)      # a state forgets what was before
    norm = (1 + rnd(g, Dv, std=0.2)).float()
    state = torch.zeros(1, H, D, Dv, device=DEV)
    x = rows.double()
    q, key = (x[:, cols[i]:cols[i] + H * D].view(n, H, D) for i in (0, 1))
    v, gate = (x[:, cols[i]:cols[i] + H * Dv].view(n, H, Dv) for i in (2, 3))
    o = (q * key).sum(-1, keepdim=True) * D ** -0.5 * v
    ref = o * torch.rsqrt((o * o).mean(-1, keepdim=True) + eps) * norm.double() * torch.nn.functional.silu(gate)
    y = k.gla_recurrent(rows.to(DEV), cols, a2.to(DEV), bias.to(DEV), norm.to(DEV), H, D, Dv, 1.0, D ** -0.5, eps,
                        context(DEV, [n], [0]), LayerCache(state=state)).double().cpu().view(n, H, Dv)
    # the sum over D may cancel: 18 roundings of its terms' sizes beside it, which the norm passes on at most whole
    spread = 18 * 2.0 ** -24 * (q * key).abs().sum(-1, keepdim=True) / (q * key).sum(-1, keepdim=True).abs()
    assert bool(((y - ref).abs() <= (2.0 ** -8 + spread) * ref.abs() + 1e-30).all()), float((y - ref).abs().max())


# narrow and wide values, rows that do not divide by the groups of threads, the most rows a thread takes; value widths that
# are no power of two go the general way
@pytest.mark.parametrize("op", ["gla", "hgrn", "ssd", "decay", "bonus"])
@pytest.mark.parametrize("H,D,Dv", [(3, 7, 16), (2, 128, 256), (1, 512, 16), (2, 100, 32), (3, 128, 128), (2, 33, 64), (2, 40, 20)])
def test_steps_of_one_token_are_the_portion_walked_along(op, H, D, Dv):
    """As above, with the sums over a column in another order: relative 2^-23 a term."""
    from simple_inference_amd.kernels import HipKernels

    if op == "bonus":
        D = Dv if Dv & (Dv - 1) == 0 else D
        Dv = D
    k = HipKernels()
    g = torch.Generator().manual_seed(H * D)
    lengths = [9, 1, 6]
    rows = projected(g, sum(lengths), H, D, Dv)
    one, state, _ = run(op, k, rows, H, D, Dv, lengths, 1)
    whole, want, _ = run(op, k, rows, H, D, Dv, lengths, 10 ** 6)
    assert float((state - want).abs().max()) <= 2e-6 * float(want.abs().max())
    assert bool(((one - whole).abs() <= 2.0 ** -7 * whole.abs() + 1e-3 * float(whole.std())).all()), float((one - whole).abs().max())


@pytest.mark.parametrize("dtype,lengths,H,D,Dv", [
    ("float32", [1000], 24, 128, 128), ("bfloat16", [1] * 200, 24, 128, 128), ("bfloat16", [300] * 40, 24, 128, 128),
    ("bfloat16", [1000], 4, 264, 64), ("bfloat16", [1000], 4, 64, 30), ("bfloat16", [100, 100], 4, 64, 64),
    ("bfloat16", [2 ** 20], 1, 8, 512), ("bfloat16", [2048], 24, 128, 128), ("bfloat16", [16384], 24, 128, 128),
    ("bfloat16", [449] + [1] * 63, 24, 128, 128)])
def test_a_step_that_is_not_cut_asks_for_no_room_for_segments(dtype, lengths, H, D, Dv):
    """The workspace is the decays and the raw outputs alone where the step is not cut: float32, one token a sequence,
    enough sequences to fill the chip, states and widths the walk does not take, portions, more segments than a grid has
    places; and a state a segment (of 64 tokens, or 128 in a long step), with no more than one further a sequence or a
    segment, where it is."""
    from simple_inference_amd.kernels import HipKernels, _DT

    core = HipKernels().core
    n, kind, cut = sum(lengths), _DT[getattr(torch, dtype)], lengths in ([2048], [16384], [449] + [1] * 63)
    facts = (n, len(lengths), max(lengths), H, D)
    segment = 128 if n * H * 2 // 128 >= 768 else 64
    room = (-(-n // segment) + min(len(lengths) - 1, -(-n // segment))) * H * D * Dv if cut else 0
    assert core.sia_gla_workspace(*facts, Dv, kind) == n * H * (D + Dv) + room
    assert core.sia_hgrn2_workspace(*facts, Dv, kind) == core.sia_ssd_workspace(*facts, Dv, kind) == n * H * (2 * D + Dv) + room
    if D == Dv:
        assert core.sia_bonus_recurrence_workspace(*facts, kind) == n * H * D + room
