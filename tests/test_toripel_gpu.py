"""Toripel on the GPU against the plain implementation (tests/plain/toripel_plain.py): the kernels of
each mechanism alone (the step of a stream of several copies, the norm a head, the passes around
attention over a latent, the product a head, the delta rule with its convolutions over unequal
requests in several steps, the experts that a table names), one-layer models of each mixer and of
the feed-forward, whole prompts against token-by-token decoding and portions down to two tokens,
mixed batches against each request alone with pages and slots that are freed and used again, keys
just inside and just outside every window in prompts, portions and decoding (with controls that a
window one off or a lost sink moves the plain logits by many times the bound), a far token that
only the delta rule's state still holds, the first tokens, long decoding through replayed graphs,
generation through the scheduler, and the trace replay program."""

from __future__ import annotations

import copy
import json
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest
import torch

from helpers import feed, make_mixed_trace, max_live_tokens, random_tokens, rel_err, replay_in_process
from plain import toripel_plain as plain
from toripel_cases import CASES, SINGLE, bare, config, delta, latent, make_tensors, tabled, windowed, write_model

pytestmark = pytest.mark.gpu
ROOT = Path(__file__).resolve().parent.parent
F64 = torch.float64

# Bounds on max |engine - plain| / max |plain logit| over a request, some three times the largest error
# measured on the MI355X on these weights (32-bit: below 6e-6 everywhere; bfloat16: 1.6e-2 on the peaked
# attention of the windows' edges, below 1.5e-2 elsewhere).
TOL = {"float32": 1.5e-5, "bfloat16": 4e-2}


def K():
    from lockstep_amd.ops import kernels
    return kernels()


@pytest.fixture(scope="module")
def models(tmp_path_factory):
    """(case, dtype) -> (loaded model, plain model, raw config, page size, folder), made once."""
    made = {}

    def get(name, dtype="float32", table=CASES, seed=11):
        from lockstep_amd import load_model

        key = (name, dtype, seed)
        if key not in made:
            case = table[name]
            tensors = make_tensors(case["raw"], seed=seed)
            folder = write_model(tmp_path_factory.mktemp(f"toripel{name}"), case["raw"], tensors)
            made[key] = (load_model(folder, dtype=dtype), plain.PlainToripel(case["raw"], tensors), case["raw"],
                         case["page_size"], folder)
        return made[key]

    return get


def new_cache(model, page_size, tokens=512, requests=4, poison=True):
    return model.make_cache(num_pages=-(-tokens // page_size), page_size=page_size, max_requests=requests,
                            max_tokens_per_request=tokens, poison_on_free=poison)


def step_meta(lengths, starts, slots):
    """tok_seq, tok_pos, seqs [n, 8] as the engine's upload lays them out."""
    seqs, tok_seq, tok_pos, off = [], [], [], 0
    for i, (n, s, slot) in enumerate(zip(lengths, starts, slots)):
        seqs.append([off, n, s, s + n, slot, 0, 0, 0])
        tok_seq += [i] * n
        tok_pos += list(range(s, s + n))
        off += n
    as_dev = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    return as_dev(tok_seq), as_dev(tok_pos), as_dev(seqs).reshape(-1)


def close(got, want, dtype, scale=1.0):
    tol = 1e-5 if dtype == torch.float32 else 1.6e-2
    return float((got.double().cpu() - want).abs().max()) <= tol * max(scale, float(want.abs().max()))


# ---------------------------------------------------------------------------
# the kernels of each mechanism alone
# ---------------------------------------------------------------------------

@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("copies, width, rows", [(1, 32, 3), (3, 100, 5), (4, 1030, 2), (8, 64, 70)])
def test_the_step_of_a_stream_of_several_copies(dtype, copies, width, rows):
    """Write alone, read alone, both in one launch, with a row list; against the plain functions."""
    g = torch.Generator().manual_seed(copies * width)
    x = torch.randn((rows, copies, width), generator=g, dtype=F64)
    partials = torch.randn((3, rows, width), generator=g, dtype=F64)
    mix, gain, take = (torch.randn(s, generator=g, dtype=F64) for s in ((copies, copies), (copies,), (copies,)))
    weight = torch.randn(width, generator=g, dtype=F64)
    f32 = lambda t: t.to(torch.float32).cuda().contiguous()  # noqa: E731
    written = plain.write_streams(x.float().double(), partials.float().double().sum(0), mix.float().double(), gain.float().double())
    want = plain.rms(plain.read_streams(written, take.float().double()), 1e-5) * weight.float().double()
    k = K()
    # both at once
    dev = f32(x).view(rows, copies * width).clone()
    out = torch.empty((rows, width), dtype=dtype, device="cuda")
    k.streams_step(dev, copies, f32(partials), f32(mix).view(-1), f32(gain), f32(take), f32(weight), 1e-5, out)
    assert close(dev.view(rows, copies, width), written, torch.float32)
    assert close(out, want, dtype)
    # the write alone, then the plain sum read for two listed rows
    dev2 = f32(x).view(rows, copies * width).clone()
    k.streams_step(dev2, copies, f32(partials), f32(mix).view(-1), f32(gain), None, None, 0.0, None)
    assert torch.equal(dev2, dev)
    listed = torch.tensor([rows - 1, 0], dtype=torch.int32, device="cuda")
    out2 = torch.empty((2, width), dtype=dtype, device="cuda")
    k.streams_step(dev2, copies, None, None, None, None, f32(weight), 1e-5, out2, listed)
    summed = plain.rms(written.sum(1), 1e-5) * weight.float().double()
    assert close(out2, summed[[rows - 1, 0]], dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("copies, width", [(1, 1024), (1, 1025), (4, 1023), (4, 1028), (6, 1024), (6, 2052), (7, 1024), (7, 1028), (8, 1020), (8, 1030)])
@pytest.mark.parametrize("centred", [False, True])
def test_the_step_of_the_copies_at_the_edges_of_a_row_of_one_run(dtype, copies, width, centred):
    """Rows of up to 1,024 elements are one run of a thread and have an instance of their own; longer ones ask for their first run
    ahead, up to six copies.  Nine slices are one more than a batch."""
    g = torch.Generator().manual_seed(copies * width + centred)
    rows = 3
    x, partials = torch.randn((rows, copies, width), generator=g), torch.randn((9, rows, width), generator=g)
    mix, gain, take = (torch.randn(s, generator=g) for s in ((copies, copies), (copies,), (copies,)))
    weight, bias = torch.randn(width, generator=g), torch.randn(width, generator=g)
    written = plain.write_streams(x.double(), partials.double().sum(0), mix.double(), gain.double())
    read = plain.read_streams(written, take.double())
    if centred:
        read = read - read.mean(-1, keepdim=True)
    want = plain.rms(read, 1e-5) * weight.double() + bias.double()
    dev = x.view(rows, copies * width).cuda().clone()
    out = torch.empty((rows, width), dtype=dtype, device="cuda")
    K().streams_step(dev, copies, partials.cuda(), mix.view(-1).cuda(), gain.cuda(), take.cuda(), weight.cuda(), 1e-5, out,
                     bias=bias.cuda(), centred=centred)
    assert close(dev.view(rows, copies, width), written, torch.float32)
    assert close(out, want, dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads, n, kk, rows", [(3, 20, 12, 5), (4, 64, 32, 130), (1, 7, 100, 17), (6, 36, 10, 66)])
def test_a_product_a_head(dtype, heads, n, kk, rows):
    g = torch.Generator().manual_seed(heads * n + kk)
    x = torch.randn((rows, heads * kk + 3), generator=g).to(dtype)
    w = torch.randn((heads, n, kk), generator=g).to(dtype)
    out = torch.zeros((rows, heads * (n + 5)), dtype=dtype, device="cuda")
    K().heads_product(x.cuda(), kk, w.cuda(), out, n + 5)
    want = torch.einsum("hnk,thk->thn", w.double(), x[:, :heads * kk].double().view(rows, heads, kk))
    got = out.view(rows, heads, n + 5)
    assert close(got[:, :, :n], want, dtype)
    assert float(got[:, :, n:].abs().max()) == 0.0          # (nothing beyond a head's columns is touched)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads, n, kk, rows", [(2, 20, 8, 5), (3, 64, 136, 16), (2, 72, 40, 64), (2, 33, 264, 130)])
def test_a_product_a_head_of_aligned_rows_has_the_bits_of_others(dtype, heads, n, kk, rows):
    """Aligned rows are read by buffer loads, rows an odd number of elements apart one element at a time: columns, rows and
    contractions that end inside a block."""
    g = torch.Generator().manual_seed(heads * n + kk)
    x = torch.randn((rows, heads * kk), generator=g).to(dtype).cuda()
    apart = torch.zeros((rows, heads * kk + 3), dtype=dtype, device="cuda")
    apart[:, :heads * kk] = x
    w = torch.randn((heads, n, kk), generator=g).to(dtype).cuda()
    out, want = (torch.zeros((rows, heads * n), dtype=dtype, device="cuda") for _ in range(2))
    K().heads_product(x, kk, w, out, n)
    K().heads_product(apart, kk, w, want, n)
    assert torch.equal(out, want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_the_passes_around_attention_over_a_latent(dtype):
    """Norms of both latents, the shared key part rotated into the pages at the tokens' positions, the queries'
    rotated part behind the latent's dimensions; two requests at different positions on scattered pages."""
    from lockstep_amd.config.base import PartSpec
    from lockstep_amd.parts import build_part

    q_rank, kv_rank, rot_dim, rot, heads, dim, page = 20, 12, 10, 6, 3, 7, 4
    dk = 24
    lengths, starts, slots = [5, 3], [6, 0], [1, 0]
    tok_seq, tok_pos, seqs = step_meta(lengths, starts, slots)
    t = sum(lengths)
    g = torch.Generator().manual_seed(5)
    raw = torch.randn((t, q_rank + kv_rank + rot_dim), generator=g)
    wq, wc = torch.randn(q_rank, generator=g), torch.randn(kv_rank, generator=g)
    position = build_part(PartSpec("rope_ramped", {"rotary_dim": rot, "theta": 50.0, "pairing": "neighbours",
                                                   "scaling": {"factor": 4.0, "original": 16, "fast": 4.0, "slow": 1.0}}))

    class RT:
        device = torch.device("cuda")
    position.ensure(16, RT)
    table = torch.tensor([[5, 1, -1, -1], [2, 0, 3, -1]], dtype=torch.int32, device="cuda")
    keys = torch.full((6, 1, page, dk), float("nan"), dtype=dtype, device="cuda")
    values = torch.full((6, 1, kv_rank, page), float("nan"), dtype=dtype, device="cuda")
    q_latent = torch.empty((t, q_rank), dtype=dtype, device="cuda")
    k = K()
    k.latent_post(raw.cuda(), t, q_rank, kv_rank, rot_dim, dk, True, wq.cuda(), wc.cuda(), 1e-5, position.cos, position.sin, rot,
                  10, tok_seq, tok_pos, seqs, table, q_latent, keys, values, page)
    f, magnitude = plain.stretched_frequencies(rot, 50.0, {"factor": 4.0, "original": 16, "fast": 4.0, "slow": 1.0})
    positions = tok_pos.cpu().long()
    want_q = plain.rms(raw[:, :q_rank].double(), 1e-5) * wq.double()
    want_c = plain.rms(raw[:, q_rank:q_rank + kv_rank].double(), 1e-5) * wc.double()
    want_r = plain.rotate_pairs(raw[:, q_rank + kv_rank:].double(), positions, f, magnitude)
    assert close(q_latent, want_q, dtype)
    rows = {1: [2, 0, 3], 0: [5, 1]}
    for i in range(t):
        slot = slots[int(tok_seq[i])]
        pos = int(tok_pos[i])
        page_id = rows[slot][pos // page]
        assert close(keys[page_id, 0, pos % page, :kv_rank], want_c[i], dtype), i
        assert close(values[page_id, 0, :, pos % page], want_c[i], dtype), i
        assert close(keys[page_id, 0, pos % page, kv_rank:kv_rank + rot_dim], want_r[i], dtype), i
        assert float(keys[page_id, 0, pos % page, kv_rank + rot_dim:].float().abs().max()) == 0.0
    # the queries: plain parts apart, rotated parts behind the latent's dimensions
    qf = torch.randn((t, heads * (dim + rot_dim)), generator=g)
    plain_out = torch.empty((t, heads * dim), dtype=dtype, device="cuda")
    q = torch.full((t, heads * dk), float("nan"), dtype=dtype, device="cuda")
    k.latent_query(qf.cuda(), t, heads, dim, rot_dim, kv_rank, dk, position.cos, position.sin, rot, 10, tok_pos, plain_out, q)
    per_head = qf.double().view(t, heads, dim + rot_dim)
    assert close(plain_out.view(t, heads, dim), per_head[:, :, :dim], dtype)
    got = q.view(t, heads, dk)
    assert close(got[:, :, kv_rank:kv_rank + rot_dim], plain.rotate_pairs(per_head[:, :, dim:], positions, f, magnitude), dtype)
    assert float(got[:, :, kv_rank + rot_dim:].float().abs().max()) == 0.0


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads, dim, rot_dim, rot, kv_rank, dk", [(3, 8, 12, 6, 12, 28), (16, 128, 64, 64, 128, 192), (5, 4, 4, 4, 4, 8),
                                                                   (7, 12, 8, 2, 8, 16), (3, 8, 10, 6, 12, 24)])
def test_latent_queries_by_whole_vectors_and_one_by_one(dtype, heads, dim, rot_dim, rot, kv_rank, dk):
    """Sizes of whole vectors of four take four elements a thread (rotated pairs that end inside a vector among them), others, and rows off a
    vector's boundary, one: the same bits, and the plain rotation."""
    t = 9
    g = torch.Generator().manual_seed(heads + dk)
    qf = torch.randn((t, heads * (dim + rot_dim)), generator=g)
    tok_pos = torch.randint(0, 30, (t,), generator=g).to(torch.int32).cuda()
    f = 50.0 ** (-torch.arange(rot // 2, dtype=torch.float64) * 2.0 / rot)
    angle = torch.arange(32, dtype=torch.float64)[:, None] * f
    cos, sin = angle.cos().float().cuda(), angle.sin().float().cuda()
    results = []
    for offset in (0, 1):
        plain_buf = torch.full((t * heads * dim + offset,), float("nan"), dtype=dtype, device="cuda")
        plain_out = plain_buf[offset:].view(t, heads * dim)
        q = torch.full((t, heads * dk), float("nan"), dtype=dtype, device="cuda")
        K().latent_query(qf.cuda(), t, heads, dim, rot_dim, kv_rank, dk, cos, sin, rot, 31, tok_pos, plain_out, q)
        results.append((plain_out.clone(), q.view(t, heads, dk)[:, :, kv_rank:].clone()))
        assert bool(torch.isnan(q.view(t, heads, dk)[:, :, :kv_rank]).all())     # (another product's place)
    assert torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][1], results[1][1])
    per_head = qf.double().view(t, heads, dim + rot_dim)
    assert close(results[0][0].view(t, heads, dim), per_head[:, :, :dim], dtype)
    assert float(results[0][1][:, :, rot_dim:].float().abs().max() if dk > kv_rank + rot_dim else 0.0) == 0.0
    assert close(results[0][1][:, :, :rot_dim], plain.rotate_pairs(per_head[:, :, dim:], tok_pos.cpu().long(), f, 1.0), dtype)


@pytest.mark.parametrize("heads, groups, d, dv, taps", [(4, 2, 24, 16, 3), (1, 1, 16, 70, 5), (3, 1, 8, 8, 1), (2, 2, 130, 20, 2),
                                                        (2, 1, 64, 33, 4)])
def test_the_delta_rule_with_its_convolutions_over_unequal_requests_in_steps(heads, groups, d, dv, taps):
    """Three requests cut into steps of unequal portions (down to one token, shorter than the taps) with their own
    state slots, against the plain convolution and recurrence over the whole sequences."""
    g = torch.Generator().manual_seed(heads * d + dv)
    channels = 2 * groups * d + heads * dv
    width = channels + 2 * heads
    lengths = {0: 23, 2: 9, 3: 40}                         # state slot -> tokens
    raws = {s: torch.randn((n, width), generator=g) for s, n in lengths.items()}
    conv = torch.randn((channels, taps), generator=g) * 0.5
    a_log, dt_bias = torch.randn(heads, generator=g) * 0.5 - 0.5, torch.randn(heads, generator=g) * 0.5
    want = {}
    for s, raw in raws.items():
        x = plain.silu(plain.short_convolution(raw[:, :channels].double(), conv.double()))
        n = raw.shape[0]
        q, kk = x[:, :groups * d].view(n, groups, d), x[:, groups * d:2 * groups * d].view(n, groups, d)
        v = x[:, 2 * groups * d:].view(n, heads, dv)
        q = q / torch.sqrt((q * q).sum(-1, keepdim=True) + 1e-6) * d ** -0.5
        kk = kk / torch.sqrt((kk * kk).sum(-1, keepdim=True) + 1e-6)
        spread = torch.arange(heads) // (heads // groups)
        beta = torch.sigmoid(raw[:, channels:channels + heads].double())
        decay = torch.exp(-torch.exp(a_log.double()) * plain.softplus(raw[:, channels + heads:].double() + dt_bias.double()))
        want[s] = plain.gated_delta_rule(q[:, spread], kk[:, spread], v, beta, decay).reshape(n, heads * dv)
    k = K()
    state = torch.zeros((5, heads * d * dv + (taps - 1) * channels), dtype=torch.float32, device="cuda")
    state[1].fill_(float("nan"))                            # (a slot that no request of the test has)
    done = {s: 0 for s in lengths}
    got = {s: [] for s in lengths}
    portions = [{0: 1, 3: 7}, {0: 2, 2: 9, 3: 1}, {0: 20, 3: 30}, {3: 2}]
    for portion in portions:
        order = list(portion)
        tok_seq, tok_pos, seqs = step_meta([portion[s] for s in order], [done[s] for s in order], order)
        raw = torch.cat([raws[s][done[s]:done[s] + portion[s]] for s in order]).cuda()
        out = torch.empty((raw.shape[0], heads * dv), dtype=torch.float32, device="cuda")
        scratch = torch.empty(k.delta_scratch_floats(raw.shape[0], groups, heads, d, dv), dtype=torch.float32, device="cuda")
        k.delta_rule(raw, groups, heads, d, dv, conv.cuda(), a_log.cuda(), dt_bias.cuda(), 1e-6, tok_seq, tok_pos, seqs,
                     len(order), state, scratch, out)
        at = 0
        for s in order:
            got[s].append(out[at:at + portion[s]].cpu())
            at += portion[s]
            done[s] += portion[s]
    assert done == lengths
    for s in lengths:
        assert close(torch.cat(got[s]), want[s], torch.float32, scale=1e-2), s


@pytest.mark.parametrize("heads, groups, d, dv, taps", [(1, 1, 250, 4, 9), (2, 1, 16, 5, 2), (1, 1, 64, 3, 4), (3, 3, 128, 16, 6)])
def test_the_delta_rule_keeps_the_last_inputs_of_every_channel(heads, groups, d, dv, taps):
    """The inputs that a step leaves for the next one's convolutions, exactly: more channels than a request has lanes, more
    taps than are moved at once, steps shorter than the taps, a request that sits a step out."""
    g = torch.Generator().manual_seed(d + taps)
    k, channels = K(), 2 * groups * d + heads * dv
    conv, a_log, dt_bias = torch.randn((channels, taps), generator=g).cuda(), torch.zeros(heads).cuda(), torch.zeros(heads).cuda()
    conv_at = heads * d * dv
    state = torch.zeros((3, conv_at + (taps - 1) * channels), dtype=torch.float32, device="cuda")
    seen = {s: torch.zeros(taps - 1, channels) for s in (0, 2)}
    done = {0: 0, 2: 0}
    for portion in ({0: 1, 2: 7}, {2: 2}, {0: 3, 2: 1}, {0: 20, 2: 1}, {0: 1, 2: 1}):
        order = list(portion)
        tok_seq, tok_pos, seqs = step_meta([portion[s] for s in order], [done[s] for s in order], order)
        raws = [torch.randn((portion[s], channels + 2 * heads), generator=g) for s in order]
        out = torch.empty((sum(portion.values()), heads * dv), dtype=torch.float32, device="cuda")
        scratch = torch.empty(k.delta_scratch_floats(len(out), groups, heads, d, dv), dtype=torch.float32, device="cuda")
        k.delta_rule(torch.cat(raws).cuda(), groups, heads, d, dv, conv, a_log, dt_bias, 1e-6, tok_seq, tok_pos, seqs, len(order), state,
                     scratch, out)
        for s, raw in zip(order, raws):
            seen[s] = torch.cat([seen[s], raw[:, :channels]])
            done[s] += portion[s]
        for s in seen:
            assert torch.equal(state[s, conv_at:].cpu().view(taps - 1, channels), seen[s][-(taps - 1):]), (portion, s)
    assert not state[1].any()


@pytest.mark.parametrize("heads, groups, d, dv", [(2, 1, 16, 17), (2, 2, 30, 5), (1, 1, 64, 64), (4, 2, 128, 20), (1, 1, 200, 9)])
@pytest.mark.parametrize("channel_decays", [False, True])
def test_the_delta_rule_has_the_same_bits_however_many_tokens_a_step_brings(heads, groups, d, dv, channel_decays):
    """Requests of every length around the blocks of tokens whose operands are fetched together, all in one step, against
    the same tokens one and two a step (which the kernel for few tokens a request takes)."""
    lengths = [1, 2, 3, 4, 5, 7, 8, 9, 15, 16, 17, 24, 31, 33]
    g = torch.Generator().manual_seed(d + dv)
    channels = 2 * groups * d + heads * dv
    conv = (torch.randn((channels, 2), generator=g) * 0.5).cuda()
    a_log = torch.randn(heads, generator=g).cuda()
    dt_bias = torch.randn(heads * d if channel_decays else heads, generator=g).cuda()
    raws = [torch.randn((n, channels + (1 if channel_decays else 2) * heads), generator=g).cuda() for n in lengths]
    chans = [torch.randn((n, heads * d), generator=g).cuda() for n in lengths]
    k = K()

    def run(most):
        state = torch.zeros((len(lengths), heads * d * dv + channels), dtype=torch.float32, device="cuda")
        outs = [[] for _ in lengths]
        for at in range(0, max(lengths), most):
            who = [i for i, n in enumerate(lengths) if n > at]
            counts = [min(most, lengths[i] - at) for i in who]
            tok_seq, tok_pos, seqs = step_meta(counts, [at] * len(who), who)
            raw = torch.cat([raws[i][at:at + n] for i, n in zip(who, counts)])
            chan = torch.cat([chans[i][at:at + n] for i, n in zip(who, counts)]) if channel_decays else None
            out = torch.full((raw.shape[0], heads * dv), float("nan"), dtype=torch.float32, device="cuda")
            size = k.delta_scratch_floats(raw.shape[0], groups, heads, d, dv, channel_decays)
            k.delta_rule(raw, groups, heads, d, dv, conv, a_log, dt_bias, 1e-6, tok_seq, tok_pos, seqs, len(who), state,
                         torch.empty(size, dtype=torch.float32, device="cuda"), out, chan)
            for i, part in zip(who, out.split(counts)):
                outs[i].append(part)
        return [torch.cat(o) for o in outs], state

    whole, state = run(max(lengths))
    assert not torch.isnan(state).any()
    for most in (1, 2):
        outs, after = run(most)
        assert torch.equal(after, state), most
        assert all(torch.equal(a, b) for a, b in zip(outs, whole)), most


@pytest.mark.parametrize("heads, groups, d, dv", [(2, 1, 16, 17), (2, 2, 30, 5), (1, 1, 64, 64), (4, 2, 128, 20), (1, 1, 200, 9)])
@pytest.mark.parametrize("channel_decays", [False, True])
def test_the_delta_rule_has_the_same_bits_whatever_it_is_told_of_the_longest_request(heads, groups, d, dv, channel_decays):
    """Many requests of one token beside a longer one: two, four or eight tokens ahead, as the caller names the longest request
    or not; each against the longer request alone."""
    g = torch.Generator().manual_seed(d + dv)
    channels = 2 * groups * d + heads * dv
    conv = (torch.randn((channels, 2), generator=g) * 0.5).cuda()
    a_log = torch.randn(heads, generator=g).cuda()
    dt_bias = torch.randn(heads * d if channel_decays else heads, generator=g).cuda()
    k = K()

    def run(counts, raw, chan, longest):
        state = torch.zeros((len(counts), heads * d * dv + channels), dtype=torch.float32, device="cuda")
        tok_seq, tok_pos, seqs = step_meta(counts, [0] * len(counts), list(range(len(counts))))
        out = torch.full((sum(counts), heads * dv), float("nan"), dtype=torch.float32, device="cuda")
        size = k.delta_scratch_floats(sum(counts), groups, heads, d, dv, channel_decays)
        k.delta_rule(raw, groups, heads, d, dv, conv, a_log, dt_bias, 1e-6, tok_seq, tok_pos, seqs, len(counts), state,
                     torch.empty(size, dtype=torch.float32, device="cuda"), out, chan, longest)
        return out, state

    for long in (2, 3, 5, 9, 13):
        counts = [1] * 13 + [long]
        n = sum(counts)
        raw = torch.randn((n, channels + (1 if channel_decays else 2) * heads), generator=g).cuda()
        chan = torch.randn((n, heads * d), generator=g).cuda() if channel_decays else None
        alone, after = run([long], raw[13:], chan[13:] if channel_decays else None, long)
        for told in (0, 1, long, 1000):
            out, state = run(counts, raw, chan, told)
            assert torch.equal(out[13:], alone) and torch.equal(state[13], after[0]), (long, told)


@pytest.mark.parametrize("channel_decays", [False, True])
def test_the_delta_rule_of_more_waves_than_fit_has_the_bits_of_one_token_a_step(channel_decays):
    """Keys of more than 128 (sixteen rows a lane) and more than two waves a SIMD: blocks of two tokens, requests of 1 to 9."""
    heads, groups, d, dv, k = 4, 2, 200, 68, K()
    n = 8 * k.compute_units() // (heads * 17) + 1  # requests: a wave works on four columns of a head
    lengths = [1 + i % 9 for i in range(n)]
    g = torch.Generator().manual_seed(n)
    channels = 2 * groups * d + heads * dv
    conv = (torch.randn((channels, 2), generator=g) * 0.5).cuda()
    a_log = torch.randn(heads, generator=g).cuda()
    dt_bias = torch.randn(heads * d if channel_decays else heads, generator=g).cuda()
    raws = [torch.randn((m, channels + (1 if channel_decays else 2) * heads), generator=g).cuda() for m in lengths]
    chans = [torch.randn((m, heads * d), generator=g).cuda() for m in lengths]

    def run(most):
        state = torch.zeros((n, heads * d * dv + channels), dtype=torch.float32, device="cuda")
        outs = [[] for _ in lengths]
        for at in range(0, max(lengths), most):
            who = [i for i, m in enumerate(lengths) if m > at]
            counts = [min(most, lengths[i] - at) for i in who]
            tok_seq, tok_pos, seqs = step_meta(counts, [at] * len(who), who)
            raw = torch.cat([raws[i][at:at + m] for i, m in zip(who, counts)])
            chan = torch.cat([chans[i][at:at + m] for i, m in zip(who, counts)]) if channel_decays else None
            out = torch.full((raw.shape[0], heads * dv), float("nan"), dtype=torch.float32, device="cuda")
            size = k.delta_scratch_floats(raw.shape[0], groups, heads, d, dv, channel_decays)
            k.delta_rule(raw, groups, heads, d, dv, conv, a_log, dt_bias, 1e-6, tok_seq, tok_pos, seqs, len(who), state,
                         torch.empty(size, dtype=torch.float32, device="cuda"), out, chan, max(counts))
            for i, part in zip(who, out.split(counts)):
                outs[i].append(part)
        return torch.cat([torch.cat(o) for o in outs]), state

    (whole, state), (single, after) = run(9), run(1)
    assert not torch.isnan(whole).any() and torch.equal(whole, single) and torch.equal(state, after)


@pytest.mark.parametrize("channel_decays", [False, True])
def test_the_delta_rule_writes_rows_any_distance_apart(channel_decays):
    """Output rows 256 MiB apart (a view into a wide buffer) get the bits of rows side by side."""
    heads, groups, d, dv, counts = 2, 1, 30, 5, [4, 1]
    g = torch.Generator().manual_seed(7)
    channels = 2 * groups * d + heads * dv
    conv = (torch.randn((channels, 2), generator=g) * 0.5).cuda()
    a_log = torch.randn(heads, generator=g).cuda()
    dt_bias = torch.randn(heads * d if channel_decays else heads, generator=g).cuda()
    raw = torch.randn((5, channels + (1 if channel_decays else 2) * heads), generator=g).cuda()
    chan = torch.randn((5, heads * d), generator=g).cuda() if channel_decays else None
    tok_seq, tok_pos, seqs = step_meta(counts, [0, 0], [0, 1])
    k = K()
    results = []
    for stride in (heads * dv, (1 << 26) + 2):
        out = torch.empty(4 * stride + heads * dv, device="cuda").as_strided((5, heads * dv), (stride, 1))
        state = torch.zeros((2, heads * d * dv + channels), device="cuda")
        scratch = torch.empty(k.delta_scratch_floats(5, groups, heads, d, dv, channel_decays), device="cuda")
        k.delta_rule(raw, groups, heads, d, dv, conv, a_log, dt_bias, 1e-6, tok_seq, tok_pos, seqs, 2, state, scratch, out, chan)
        results.append((out.clone(memory_format=torch.contiguous_format), state))
        del out
    torch.cuda.empty_cache()
    assert torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][1], results[1][1])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("tokens, experts, top, width, ff", [(1, 4, 2, 32, 24), (37, 7, 3, 64, 40), (300, 5, 1, 48, 16),
                                                              (700, 3, 3, 32, 8)])
def test_experts_that_a_table_names(dtype, tokens, experts, top, width, ff):
    g = torch.Generator().manual_seed(tokens + experts)
    vocab = 50
    ids = torch.randint(0, vocab, (tokens,), generator=g)
    table = torch.stack([torch.randperm(experts, generator=g)[:top] for _ in range(vocab)]).to(torch.int32)
    x = torch.randn((tokens, width), generator=g).to(dtype)
    w_gate, w_up = (torch.randn((experts, ff, width), generator=g) * 0.3).to(dtype), (torch.randn((experts, ff, width), generator=g) * 0.3).to(dtype)
    w_down = (torch.randn((experts, width, ff), generator=g) * 0.3).to(dtype)
    want = plain.tabled_experts(x.double(), ids, table.long(),
                                [(w_gate[e].double(), w_up[e].double(), w_down[e].double()) for e in range(experts)])
    k = K()
    rows = 16 if tokens * top / experts <= 16 else 32 if tokens * top / experts <= 64 else 64
    cap = k.experts_tile_capacity(tokens, experts, top, rows)
    i32 = lambda n: torch.empty(n, dtype=torch.int32, device="cuda")  # noqa: E731
    chosen, order, tiles, counts = i32(tokens * top), i32(tokens * top), i32(4 * cap), i32(experts)
    share = torch.empty(tokens * top, dtype=torch.float32, device="cuda")
    k.experts_route_table(ids.to(torch.int32).cuda(), table.cuda(), experts, rows, chosen, share, order, tiles, counts)
    assert torch.equal(chosen.cpu().view(tokens, top), table[ids])
    act = torch.empty((tokens * top, ff), dtype=dtype, device="cuda")
    partials = torch.empty((top, tokens, width), dtype=torch.float32, device="cuda")
    k.experts_apply(x.cuda(), w_gate.cuda(), w_up.cuda(), w_down.cuda(), top, rows, order, tiles, share, float("inf"), 1.0, act,
                    partials, shift=0.0)
    assert close(partials.sum(0), want, dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("weigh_input,identity", [(False, 0), (True, 0), (False, 2)])
@pytest.mark.parametrize("tokens,experts,top,width,ff", [(1, 4, 1, 512, 512), (9, 8, 2, 1024, 768), (40, 6, 3, 1536, 2048), (17, 1, 1, 768, 16 * 48),
                                                         (150, 32, 1, 1024, 512)])
def test_experts_of_few_rows_have_the_bits_of_the_kernels_for_any_size(dtype, tokens, experts, top, width, ff, weigh_input, identity):
    """Tiles of 16 rows of whole chunks (one round and several of 4, 6 and 8; a last tile of one row; experts that return their
    input) against the kernels for any size, which a tile list off 16 bytes goes to."""
    g = torch.Generator().manual_seed(tokens + width)
    k, all_of = K(), experts + identity
    ids = torch.arange(tokens, dtype=torch.int32).cuda()
    table = torch.stack([torch.randperm(all_of, generator=g)[:top] for _ in range(tokens)]).to(torch.int32).cuda()
    x = torch.randn((tokens, width), generator=g).to(dtype).cuda()
    w_gate, w_up, w_down = ((torch.randn((experts, *s), generator=g) * s[1] ** -0.5).to(dtype).cuda() for s in ((ff, width), (ff, width), (width, ff)))
    cap = k.experts_tile_capacity(tokens, all_of, top, 16)
    outs = []
    for shift in (0, 1):
        i32 = lambda n: torch.empty(n, dtype=torch.int32, device="cuda")  # noqa: E731
        chosen, order, tiles, counts = i32(tokens * top), i32(tokens * top), i32(4 * cap + shift)[shift:], i32(all_of)
        share = torch.empty(tokens * top, dtype=torch.float32, device="cuda")
        k.experts_route_table(ids, table, all_of, 16, chosen, share, order, tiles, counts)
        share.copy_(torch.rand(tokens * top, generator=torch.Generator().manual_seed(5)))
        act = torch.zeros((tokens * top, ff), dtype=dtype, device="cuda")
        partials = torch.full((top, tokens, width), float("nan"), device="cuda")
        k.experts_apply(x, w_gate, w_up, w_down, top, 16, order, tiles, share, 3.0, 1.5, act, partials, shift=0.5, weigh_input=weigh_input,
                        identity=identity)
        assert not torch.isnan(partials).any()
        outs.append(partials)
    assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("tokens,experts,top,width,ff", [(1, 4, 1, 512, 512), (8, 32, 4, 1024, 768), (21, 6, 3, 1536, 2048), (64, 3, 1, 512, 1536),
                                                         (33, 1, 1, 768, 768), (1, 64, 64, 512, 512), (16, 300, 4, 512, 512)])
def test_few_pairs_that_a_table_names_without_a_launch_to_order_them(dtype, tokens, experts, top, width, ff):
    """Steps of up to 64 pairs (one expert's rows in one, two and four workgroups; a table that names every expert) against the
    routing and the products in launches of their own: the same bits, tokens that repeat among them."""
    g = torch.Generator().manual_seed(tokens * top + width)
    k, vocab = K(), 40
    assert k.experts_apply_table_ok(dtype, tokens, experts, top, width, ff, width)
    assert not k.experts_apply_table_ok(dtype, 64 // top + 1, experts, top, width, ff, width)
    assert not k.experts_apply_table_ok(dtype, tokens, experts, top, width + 16, ff, width)
    ids = torch.randint(0, vocab, (tokens,), generator=g).to(torch.int32).cuda()
    table = torch.stack([torch.randperm(experts, generator=g)[:top] for _ in range(vocab)]).to(torch.int32).cuda()
    x = torch.randn((tokens, width), generator=g).to(dtype).cuda()
    w_gate, w_up, w_down = ((torch.randn((experts, *s), generator=g) * s[1] ** -0.5).to(dtype).cuda() for s in ((ff, width), (ff, width), (width, ff)))
    cap = k.experts_tile_capacity(tokens, experts, top, 16)
    i32 = lambda n: torch.empty(n, dtype=torch.int32, device="cuda")  # noqa: E731
    chosen, order, tiles, counts = i32(tokens * top), i32(tokens * top), i32(4 * cap), i32(experts)
    share = torch.empty(tokens * top, dtype=torch.float32, device="cuda")
    k.experts_route_table(ids, table, experts, 16, chosen, share, order, tiles, counts)
    act = torch.full((tokens * top, ff), float("nan"), dtype=dtype, device="cuda")
    want, got = (torch.full((top, tokens, width), float("nan"), device="cuda") for _ in range(2))
    k.experts_apply(x, w_gate, w_up, w_down, top, 16, order, tiles, share, 3.0, 1.5, act, want, shift=0.5)
    act.fill_(float("nan"))
    picked = torch.full_like(chosen, -1)
    k.experts_apply_table(x, w_gate, w_up, w_down, ids, table, 3.0, 1.5, act, picked, got, shift=0.5)
    assert not torch.isnan(want).any() and torch.equal(got, want) and torch.equal(picked, chosen)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("tokens,experts,top,rows", [(1, 512, 4, 9), (7, 32, 4, 40), (33, 40, 1, 1), (63, 64, 1, 2), (16, 64, 4, 3), (21, 33, 3, 1),
                                                     (16, 4, 4, 5)])
def test_pairs_of_many_experts_that_a_table_names(dtype, tokens, experts, top, rows):
    """Fewer pairs than experts and sixteens of tokens, so that a workgroup stands for a pair: one expert's rows in one, two, three and four
    of them (a table of one row and of few), pairs in no order, one pair, as many workgroups by pairs as by experts."""
    g = torch.Generator().manual_seed(tokens * top + experts)
    k, width, ff = K(), 512, 512
    ids = torch.randint(0, rows, (tokens,), generator=g).to(torch.int32).cuda()
    table = torch.stack([torch.randperm(experts, generator=g)[:top] for _ in range(rows)]).to(torch.int32).cuda()
    x = torch.randn((tokens, width), generator=g).to(dtype).cuda()
    w_gate, w_up, w_down = ((torch.randn((experts, *s), generator=g) * s[1] ** -0.5).to(dtype).cuda() for s in ((ff, width), (ff, width), (width, ff)))
    cap = k.experts_tile_capacity(tokens, experts, top, 16)
    i32 = lambda n: torch.empty(n, dtype=torch.int32, device="cuda")  # noqa: E731
    chosen, order, tiles, counts = i32(tokens * top), i32(tokens * top), i32(4 * cap), i32(experts)
    share = torch.empty(tokens * top, dtype=torch.float32, device="cuda")
    k.experts_route_table(ids, table, experts, 16, chosen, share, order, tiles, counts)
    act = torch.full((tokens * top, ff), float("nan"), dtype=dtype, device="cuda")
    want, got = (torch.full((top, tokens, width), float("nan"), device="cuda") for _ in range(2))
    k.experts_apply(x, w_gate, w_up, w_down, top, 16, order, tiles, share, 3.0, 1.5, act, want, shift=0.5)
    act.fill_(float("nan"))
    picked = torch.full_like(chosen, -1)
    k.experts_apply_table(x, w_gate, w_up, w_down, ids, table, 3.0, 1.5, act, picked, got, shift=0.5)
    assert not torch.isnan(want).any() and torch.equal(got, want) and torch.equal(picked, chosen)


# ---------------------------------------------------------------------------
# whole models
# ---------------------------------------------------------------------------

@pytest.mark.parametrize("kind", ["windowed", "latent", "latent_wide", "delta", "tabled", "odd_width"])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_each_mechanism_alone_whole_and_in_portions(models, kind, dtype):
    model, oracle, raw, page, _ = models(kind, dtype, table=SINGLE)
    tokens = random_tokens(75, raw["vocab"], seed=4)
    want = oracle.forward(tokens)
    for cuts in ([], [2, 31, 2, 17, 1, 1, 1], [1] * 75):
        cache = new_cache(model, page)
        got = feed(model, cache, "r", tokens, cuts)
        assert rel_err(got, want) < TOL[dtype], (kind, cuts[:3])
        cache.close("r")
        cache.audit()


@pytest.mark.parametrize("name", ["A", "B", "C"])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_whole_prompt_portions_and_token_by_token_agree_with_the_plain_model(models, name, dtype):
    model, oracle, raw, page, _ = models(name, dtype)
    tokens = random_tokens(150, raw["vocab"], seed=5)
    want = oracle.forward(tokens)
    runs = {}
    for label, cuts in (("whole", []), ("portions", [2, 47, 3, 16, 2, 33, 5, 1, 1, 2]), ("tail", [110] + [1] * 40),
                        ("single", [1] * 150)):
        cache = new_cache(model, page)
        runs[label] = feed(model, cache, "r", tokens, cuts)
        assert rel_err(runs[label], want) < TOL[dtype], (name, label)
        cache.close("r")
        cache.audit()
    if dtype == "float32":              # the cuttings agree with each other far below the bound against the plain model
        for label in ("portions", "tail", "single"):
            assert rel_err(runs[label], runs["whole"]) < 1e-5, label


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_a_long_prompt_and_decoding_after_it(models, dtype):
    """A prompt of 700 tokens (many row blocks, windows that have long passed the first pages, a recurrent state
    carried over hundreds of tokens), whole and cut at odd places, and twenty decoded tokens after it."""
    model, oracle, raw, page, _ = models("A", dtype)
    tokens = random_tokens(720, raw["vocab"], seed=13)
    want = oracle.forward(tokens)
    for cuts in ([700] + [1] * 20, [333, 2, 365] + [1] * 20):
        cache = new_cache(model, page, tokens=1024)
        got = feed(model, cache, "r", tokens, cuts)
        assert rel_err(got, want) < TOL[dtype], cuts[:3]
        cache.close("r")


@pytest.mark.parametrize("name", ["A", "B", "C"])
def test_first_tokens_and_prompts_of_one_and_two_tokens(models, name):
    model, oracle, raw, page, _ = models(name)
    for n in (1, 2, 3, page, page + 1):
        tokens = random_tokens(n, raw["vocab"], seed=20 + n)
        cache = new_cache(model, page)
        assert rel_err(feed(model, cache, "r", tokens, []), oracle.forward(tokens)) < TOL["float32"], n


@pytest.mark.parametrize("name, dtype", [("A", "float32"), ("B", "float32"), ("C", "float32"), ("A", "bfloat16")])
def test_mixed_batches_of_unequal_requests_with_pages_and_slots_used_again(models, name, dtype):
    """Seven requests of unequal lengths through four slots and a pool that holds the live ones only:
    portions beside single tokens, requests that sit steps out, finished requests whose (poisoned)
    pages and state slots the next ones take.  Each request's logits equal those of the request alone."""
    model, oracle, raw, page, _ = models(name, dtype)
    lengths = [1, 23, 97, 150, 61, 2, 130]
    requests = {f"r{i}": random_tokens(n, raw["vocab"], seed=40 + i) for i, n in enumerate(lengths)}
    steps = make_mixed_trace(requests, seed=3, max_live=4, decode_tail=12, max_portion=29)
    assert any(len(s["entries"]) > 1 and {len(e["tokens"]) for e in s["entries"]} != {1} for s in steps)
    tokens = max_live_tokens(steps, round_to=page)
    cache = model.make_cache(num_pages=-(-tokens // page), page_size=page, max_requests=4,
                             max_tokens_per_request=max(lengths) + page, poison_on_free=True)
    got = replay_in_process(model, cache, steps)
    assert cache.free_slots == 4 and all(g.pool.taken_total > g.pool.num_pages for g in cache.groups)
    for rid, toks in requests.items():
        assert rel_err(got[rid], oracle.forward(toks)) < TOL[dtype], rid


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_a_model_whose_few_pairs_find_their_experts_themselves(tmp_path, monkeypatch, dtype):
    """A model wide enough for ``experts_apply_table``: a prompt in portions on both sides of the rule, a mixed batch, and two requests
    through replayed graphs, against the plain model, and with the same bits as the engine that puts the pairs in order first."""
    from lockstep_amd import load_model
    from lockstep_amd.engine.batch import StepEntry

    raw = config(512, 96, [tabled(windowed(4, 2, 32, 16, window=21, scale=0.5), 512, experts=6, top=2),
                           tabled(delta(2, 1, 32, 24, taps=3), 768, experts=40, top=3)], streams=2)
    tensors = make_tensors(raw, seed=31)
    folder, oracle = write_model(tmp_path / "m", raw, tensors), plain.PlainToripel(raw, tensors)
    kernels, calls = type(K()), []
    apply_table = kernels.experts_apply_table
    monkeypatch.setattr(kernels, "experts_apply_table", lambda self, x, *rest, **named: (calls.append(x.shape[0]), apply_table(self, x, *rest, **named))[1])
    prompt = random_tokens(140, raw["vocab"], seed=6)
    requests = {f"r{i}": random_tokens(n, raw["vocab"], seed=50 + i) for i, n in enumerate([1, 23, 61, 2, 40])}
    steps = make_mixed_trace(requests, seed=4, max_live=4, decode_tail=8, max_portion=19)
    pair = random_tokens(90, raw["vocab"], seed=8), random_tokens(80, raw["vocab"], seed=9)
    runs = {}
    for listed in (False, True):
        if listed:
            monkeypatch.setattr(kernels, "experts_apply_table_pays", lambda self, tokens, experts, top: False)
        model = load_model(folder, dtype=dtype)
        cache = new_cache(model, 8, tokens=512)
        got = [feed(model, cache, "r", prompt, [1, 3, 16, 17, 21, 22, 5, 32, 1, 8])]
        cache.close("r")
        out = replay_in_process(model, cache, steps)
        got += [out[rid] for rid in requests]
        cache.open("a"), cache.open("b")
        model.step(cache, [StepEntry("a", pair[0][:30], []), StepEntry("b", pair[1][:20], [])])
        replays, rows = model.graph_replays, []
        for t in range(60):
            rows.append(model.step(cache, [StepEntry("a", [pair[0][30 + t]], [0]), StepEntry("b", [pair[1][20 + t]], [0])]).cpu())
        assert model.graph_replays - replays >= 40
        got += [torch.stack([r[i] for r in rows]) for i in range(2)]
        runs[listed] = [torch.as_tensor(g).cpu() for g in got]
        if not listed:
            assert {1, 2, 3, 8, 16} <= set(calls) and max(calls) <= 32, sorted(set(calls))
            taken = len(calls)
        assert len(calls) == taken
    want = [oracle.forward(prompt), *(oracle.forward(toks) for toks in requests.values()), oracle.forward(pair[0])[30:], oracle.forward(pair[1])[20:]]
    for i, (mine, other, plain_rows) in enumerate(zip(runs[False], runs[True], want)):
        assert torch.equal(mine, other), i
        assert rel_err(mine, plain_rows) < TOL[dtype], i


# ---------------------------------------------------------------------------
# windows' edges, the sink, a far token
# ---------------------------------------------------------------------------

def _edge_case(kind):
    """One mixer whose attention is peaked (a large scale on normalised or enlarged queries), so that the one key
    just inside a window's edge often holds most of a row's weight."""
    if kind == "windowed":
        layer = bare(windowed(2, 1, 16, 24, window=19, scale=1.6))
    else:
        layer = bare(latent(2, 16, 8, 24, q_rank=24, kv_rank=16, window=19, scale=2.5, base=100.0))
    return config(48, 40, [layer, copy.deepcopy(layer)], streams=2)


@pytest.mark.parametrize("kind", ["windowed", "latent"])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("page", [8, 16])
def test_keys_just_inside_and_just_outside_a_window(tmp_path, kind, dtype, page):
    """Prompts, portions that end and start around the window's edge, and decoding while the window moves over
    prompt and decoded tokens.  Controls: a window one key wider or narrower, and a lost sink, move the plain
    logits by many times the bound, so an engine that agrees has neither."""
    from lockstep_amd import load_model

    raw = _edge_case(kind)
    tensors = make_tensors(raw, seed=21, spread=1.5)
    # (sinks that weigh as much as a row's best keys: a lost one moves the logits by half their size)
    tensors = {name: (t.float() + 2.0).to(t.dtype) if name.endswith(".sink") else t for name, t in tensors.items()}
    model = load_model(write_model(tmp_path / "m", raw, tensors), dtype=dtype)
    oracle = plain.PlainToripel(raw, tensors)
    tokens = random_tokens(90, raw["vocab"], seed=6)
    want = oracle.forward(tokens)
    for off in (-1, 1):
        other = copy.deepcopy(raw)
        for layer in other["layers"]:
            layer["mixer"]["mask"]["size"] += off
        assert rel_err(plain.PlainToripel(other, tensors).forward(tokens), want) > 10 * TOL[dtype], off
    if kind == "latent":
        lost = {name: (t.float() - 30.0).to(t.dtype) if name.endswith(".sink") else t for name, t in tensors.items()}
        assert rel_err(plain.PlainToripel(raw, lost).forward(tokens), want) > 10 * TOL[dtype]
    for cuts in ([], [18, 1, 1, 1, 19, 2, 17, 20, 3], [19] + [1] * 71, [1] * 90, [40] + [1] * 50):
        cache = new_cache(model, page, tokens=128)
        got = feed(model, cache, "r", tokens, cuts)
        assert rel_err(got, want) < TOL[dtype], (kind, cuts[:3])
        cache.close("r")
        cache.audit()


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_a_far_token_that_only_the_state_still_holds(tmp_path, dtype):
    """A delta layer between two windowed ones: the second token of 300 is far outside every window, and the
    logits at the end still depend on it (control), through the state that prompt portions and decoded tokens
    carried."""
    from lockstep_amd import load_model

    near = bare(windowed(2, 1, 16, 16, window=9, scale=0.5))
    raw = config(48, 40, [near, bare(delta(2, 1, 16, 24, taps=3)), copy.deepcopy(near)], streams=2)
    tensors = make_tensors(raw, seed=22, spread=1.5)
    tensors["l1.mix.A_log"] = torch.full_like(tensors["l1.mix.A_log"], -6.0)       # (a slow decay: a long memory)
    model = load_model(write_model(tmp_path / "m", raw, tensors), dtype=dtype)
    oracle = plain.PlainToripel(raw, tensors)
    tokens = random_tokens(300, raw["vocab"], seed=7)
    want = oracle.forward(tokens)
    changed = list(tokens)
    changed[1] = (tokens[1] + 1) % raw["vocab"]
    assert rel_err(oracle.forward(changed)[-20:], want[-20:]) > 100 * TOL["float32"]    # (7e-3: what the 32-bit path must show)
    for cuts in ([], [100, 2, 150] + [1] * 48, [250] + [1] * 50):
        cache = new_cache(model, 8, tokens=384)
        got = feed(model, cache, "r", tokens, cuts)
        assert rel_err(got[-20:], want[-20:]) < TOL[dtype], cuts[:3]
        assert rel_err(got, want) < TOL[dtype], cuts[:3]
        cache.close("r")


# ---------------------------------------------------------------------------
# long decoding, generation, the programs
# ---------------------------------------------------------------------------

@pytest.mark.parametrize("name", ["A", "C"])
def test_long_decoding_of_two_requests_through_replayed_graphs(models, name):
    from lockstep_amd.engine.batch import StepEntry

    model, oracle, raw, page, _ = models(name)
    a, b = random_tokens(230, raw["vocab"], seed=8), random_tokens(215, raw["vocab"], seed=9)
    cache = new_cache(model, page, tokens=512)
    cache.open("a"), cache.open("b")
    model.step(cache, [StepEntry("a", a[:30], []), StepEntry("b", b[:15], [])])
    replays = model.graph_replays
    rows = {"a": [], "b": []}
    for t in range(200):
        logits = model.step(cache, [StepEntry("a", [a[30 + t]], [0]), StepEntry("b", [b[15 + t]], [0])])
        rows["a"].append(logits[0].cpu()), rows["b"].append(logits[1].cpu())
    assert model.graph_replays - replays >= 150
    assert rel_err(torch.stack(rows["a"]), oracle.forward(a)[30:]) < TOL["float32"]
    assert rel_err(torch.stack(rows["b"]), oracle.forward(b)[15:]) < TOL["float32"]


@pytest.mark.parametrize("name", ["A", "B"])
def test_greedy_generation_through_the_scheduler_and_the_single_prompt_entry_point(models, name):
    from lockstep_amd import LLM, Request

    _, oracle, raw, page, folder = models(name, seed=12)
    prompts = [random_tokens(n, raw["vocab"], seed=60 + n) for n in (5, 41, 18)]
    want = [oracle.generate_greedy(p, 24) for p in prompts]
    llm = LLM(folder, dtype="float32", num_pages=64, page_size=page)
    got = llm.generate([Request(uid=f"r{i}", prompt=p, max_new_tokens=24) for i, p in enumerate(prompts)])
    assert [got[f"r{i}"] for i in range(3)] == want
    alone, _ = llm.generate_greedy(prompts[1], 24)
    assert alone == want[1]
    half = LLM(folder, dtype="bfloat16", num_pages=64, page_size=page)
    tokens = half.generate([Request(uid="x", prompt=prompts[0], max_new_tokens=8)])["x"]
    assert len(tokens) == 8 and tokens[:2] == want[0][:2]


def test_trace_replay_program_on_a_model_folder(models, tmp_path):
    """bin/trace_run as a subprocess on a Toripel folder: a mixed schedule through four slots."""
    _, oracle, raw, page, folder = models("A")
    requests = {f"q{i}": random_tokens(n, raw["vocab"], seed=80 + i) for i, n in enumerate([40, 3, 77, 52, 19])}
    steps = make_mixed_trace(requests, seed=5, max_live=4, decode_tail=6, max_portion=19)
    out = tmp_path / "out"
    proc = subprocess.Popen([sys.executable, str(ROOT / "bin" / "trace_run"), "--model", str(folder), "--dtype", "float32",
                             "--out", str(out), "--max-tokens", str(max_live_tokens(steps)), "--page-size", str(page)],
                            stdin=subprocess.PIPE, stdout=subprocess.PIPE, text=True)
    try:
        for step in steps:
            proc.stdin.write(json.dumps(step) + "\n")
            proc.stdin.flush()
            assert proc.stdout.readline().strip() == f"done {step['step']}"
        proc.stdin.close()
        assert proc.wait(timeout=60) == 0
    finally:
        if proc.poll() is None:
            proc.kill()
    rows: dict = {}
    for step in steps:
        data = np.fromfile(out / f"{step['step']}.f32", dtype="<f4").reshape(-1, raw["vocab"])
        at = 0
        for e in step["entries"]:
            rows.setdefault(e["id"], []).append(data[at:at + len(e["want"])])
            at += len(e["want"])
    for rid, toks in requests.items():
        assert rel_err(np.concatenate(rows[rid]), oracle.forward(toks)) < TOL["float32"], rid
