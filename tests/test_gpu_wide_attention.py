"""One wide head (heads = 1, head_dim = 512: the VAE mid-block) through the host
mirror and the C ABI, against the CPU oracle (runtime/attention.zig).

Tolerance: the bf16 attention bar, max |err| <= 2e-2 and mean |err| <= 2e-3 on
outputs of unit scale (Q, K, V rounded to bf16, fp32 accumulation); the
reference's own test of its wide kernel (metal/mattn_test.zig:138-230) uses
N(0, 0.25) inputs, the smallest multiple of 64 past 6144 tokens, sampled rows
including both row blocks of the first, a middle and the last workgroup, and
byte-equal reruns: restated here.
"""
import ctypes as C

import numpy as np
import pytest

from oracle import zoracle as zo
from tests import refimpl
from zdraw_amd import hip, host

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = host.Context.init()
    yield c
    c.deinit()


def draw(rng, tokens, scale=1.0):
    return tuple((rng.standard_normal((tokens, 1, 512), dtype=np.float32) * np.float32(scale)) for _ in range(3))


@pytest.mark.parametrize("tokens", [64, 128, 448, 1024])
def test_wide_head_matches_oracle_on_every_row(ctx, tokens):
    rng = np.random.default_rng(40 + tokens)
    q, k, v = draw(rng, tokens)
    cfg = host.Config(tokens, 1, 1, 512)
    got = ctx.run(q, k, v, cfg).reshape(tokens, 1, 512)
    want = zo.attention_run(q, k, v, zo.Config(tokens, 1, 1, 512))
    refimpl.check_close(got, want, f"wide head, {tokens} tokens")
    # pooled and caller-owned-handle forms run the same kernel: same bytes
    again = ctx.run_pooled(q, k, v, cfg).reshape(tokens, 1, 512)
    assert np.array_equal(got, again)


# The key loop walks two blocks a trip and the two waves of a pair swap their blocks' probabilities through two
# slots in turn: few blocks and no range, two ranges of nine blocks, ranges of nine and a last one of seven with
# half a query tile left over; every row, so that each wave's half of the dims counts.
@pytest.mark.parametrize("tokens", [192, 576, 1088])
def test_wide_head_odd_numbers_of_blocks_on_every_row(ctx, tokens):
    rng = np.random.default_rng(60 + tokens)
    q, k, v = draw(rng, tokens)
    got = ctx.run(q, k, v, host.Config(tokens, 1, 1, 512)).reshape(tokens, 1, 512)
    want = zo.attention_run(q, k, v, zo.Config(tokens, 1, 1, 512))
    refimpl.check_close(got, want, f"wide head, {tokens} tokens")


# Rows whose scores against the first block of a key range are infinite or no numbers: the reference point is
# taken from that block and starts every score behind it, so nothing of such a row may be used as it stands (its tile is formed
# again with a running maximum). -inf: those keys weigh nothing. +inf, NaN: the row is NaN, as in the
# oracle. The rows between them, and the tiles beside theirs, are ordinary. One range; two of nine blocks.
@pytest.mark.parametrize("tokens", [256, 576])
@pytest.mark.parametrize("kind", ["-inf", "+inf", "nan"])
def test_wide_head_first_block_without_a_finite_maximum(ctx, tokens, kind):
    rng = np.random.default_rng(70 + tokens)
    q, k, v = draw(rng, tokens)
    odd = np.zeros(tokens, bool)
    odd[1:128:2] = True  # rows of the first tile
    q[~odd, :, 0] = 0.0
    k[:, :, 0] = 0.0
    q[odd, :, 0] = np.float32("nan") if kind == "nan" else np.float32(2.0 ** 100)
    for first in {0, 32 * (tokens // 64)} if kind != "nan" else ():
        k[first:first + 32, :, 0] = np.float32(2.0 ** 60) * (1 if kind == "+inf" else -1)  # products of 2^160
    got = ctx.run(q, k, v, host.Config(tokens, 1, 1, 512)).reshape(tokens, 1, 512)
    want = zo.attention_run(q, k, v, zo.Config(tokens, 1, 1, 512))
    refimpl.check_close(got[~odd], want[~odd], f"wide head, rows beside those with {kind}")
    if kind == "-inf":
        refimpl.check_close(got[odd], want[odd], "wide head, first blocks at -inf")
    else:
        assert np.isnan(want[odd]).all() and np.isnan(got[odd]).all()


# Numbers of key blocks that the number of ranges does not divide (the last range is shorter),
# half a query tile left over, three to seven ranges, and both sides of the length
# where two ranges a tile outgrow one round; rows of the first, a middle and the last tile.
@pytest.mark.parametrize("tokens", [704, 1344, 1984, 3008, 8256, 16448])
def test_wide_head_uneven_key_ranges_sampled_rows_and_rerun(ctx, tokens):
    rng = np.random.default_rng(90 + tokens)
    q, k, v = draw(rng, tokens)
    cfg = host.Config(tokens, 1, 1, 512)
    got = ctx.run(q, k, v, cfg).reshape(tokens, 1, 512)
    again = ctx.run(q, k, v, cfg).reshape(tokens, 1, 512)
    assert got.tobytes() == again.tobytes()
    rows = [0, 31, 127, tokens // 2, tokens - 65, tokens - 64, tokens - 1]
    want = zo.attention_token_list(q, k, v, zo.Config(tokens, 1, 1, 512), rows)
    refimpl.check_close(got[rows], want.reshape(len(rows), 1, 512), f"wide head, {tokens} tokens")
    assert (np.abs(got).max(axis=(1, 2)) > 0).all()


# Lengths whose number of ranges rests on how the estimate rises with the fill of a round: six ranges with a last one of
# four blocks, seven with one of two, eight of ten each, four that nearly fill a round, five over two rounds and a half.
@pytest.mark.parametrize("tokens,want", [(1408, 6), (1600, 7), (2560, 8), (7424, 4), (16640, 5)])
def test_wide_head_ranges_by_the_fill_of_a_round(ctx, tokens, want):
    n, share = C.c_uint32(0), C.c_uint64(0)
    hip.lib().zdraw_hip_wide_ranges(tokens, 256, C.byref(n), C.byref(share))
    assert n.value == want
    test_wide_head_uneven_key_ranges_sampled_rows_and_rerun(ctx, tokens)


def test_wide_head_reference_case_sampled_rows_and_rerun(ctx):
    # metal/mattn_test.zig:138-230
    tokens = 6208
    rng = np.random.default_rng(0x51DE)
    q, k, v = draw(rng, tokens, 0.5)
    cfg = host.Config(tokens, 1, 1, 512)
    got = ctx.run(q, k, v, cfg).reshape(tokens, 1, 512)
    again = ctx.run(q, k, v, cfg).reshape(tokens, 1, 512)
    assert got.tobytes() == again.tobytes()
    assert np.isfinite(got).all()
    ocfg = zo.Config(tokens, 1, 1, 512)
    rows = [0, 7, 8, 15, 16, 31, 32, 63, 64, 3103, 6191, 6207]
    want = zo.attention_token_list(q, k, v, ocfg, rows)
    err = np.abs(got[rows] - want.reshape(len(rows), 1, 512))
    # the reference's bar for its half-precision MMA kernel on these inputs is 2e-3 absolute
    assert err.max() <= 2e-3, err.max()
    # every row is written: with 6208 keys of N(0, 0.25) values no output row can be exactly zero
    assert (np.abs(got).max(axis=(1, 2)) > 0).all()


def test_wide_head_at_the_1024_px_length_sampled_rows_and_rerun(ctx):
    # 16384 tokens, the VAE mid-block of a 1024 px render and the length the kernel's throughput
    # is quoted on: one workgroup per CU, no key ranges. Sampled rows in the manner of
    # metal/mattn_test.zig:138-224 (both halves of the first, a middle and the last query tile,
    # rows of every wave), N(0, 1) operands at the bf16 bar, byte-equal rerun.
    tokens = 16384
    rng = np.random.default_rng(0x16384)
    q, k, v = draw(rng, tokens)
    cfg = host.Config(tokens, 1, 1, 512)
    got = ctx.run(q, k, v, cfg).reshape(tokens, 1, 512)
    again = ctx.run(q, k, v, cfg).reshape(tokens, 1, 512)
    assert got.tobytes() == again.tobytes()
    assert np.isfinite(got).all()
    rows = [0, 31, 32, 63, 64, 95, 96, 127, 128, 8191, 8192, 8255, 12345, 16256, 16319, 16352, 16383]
    want = zo.attention_token_list(q, k, v, zo.Config(tokens, 1, 1, 512), rows)
    refimpl.check_close(got[rows], want.reshape(len(rows), 1, 512), "wide head, 16384 tokens")
    assert (np.abs(got).max(axis=(1, 2)) > 0).all()


def test_wide_head_sharp_softmax_and_large_scores(ctx):
    # rows whose scores span a wide range (no QK-norm in front of this attention): a key along
    # the query's direction scores about 34 against a field of N(0, 1) scores; the running
    # maximum must follow it wherever in the sequence it sits (first block, last block, middle),
    # and the blocks far below it must contribute next to nothing. (The planted keys are kept
    # moderate: a bf16 operand's rounding error grows with the score, for every other row too.)
    tokens = 256
    rng = np.random.default_rng(77)
    q, k, v = draw(rng, tokens)
    for i, j in ((3, 0), (40, 255), (200, 100)):
        k[j, 0] = 1.5 * q[i, 0] / np.linalg.norm(q[i, 0]) * np.sqrt(512.0)
    got = ctx.run(q, k, v, host.Config(tokens, 1, 1, 512)).reshape(tokens, 1, 512)
    want = zo.attention_run(q, k, v, zo.Config(tokens, 1, 1, 512))
    refimpl.check_close(got, want, "sharp softmax")
    for i, j in ((3, 0), (40, 255), (200, 100)):
        assert np.abs(want[i, 0] - v[j, 0]).max() < 1e-3  # the planted key really takes the whole row


def test_wide_head_rows_overtaken_several_times_within_reach(ctx):
    # 1152 tokens (nine query tiles, 36 key blocks): rows whose best key so far is overtaken
    # three times, 8 to 11 in the score each time (each planted key keeps e^-8 .. e^-11 of the
    # weight of the next): within reach of the reference point, the first block's maximum, which
    # stays where it is while the P of these keys grow to 2^40; rows in every wave of a tile and
    # in both halves of the output dims are checked against the oracle like all others.
    tokens = 1152
    rng = np.random.default_rng(78)
    q, k, v = draw(rng, tokens)
    rows = (5, 37, 70, 127, 600, 1151)
    for n, i in enumerate(rows):
        unit = q[i, 0] / np.linalg.norm(q[i, 0]) * np.sqrt(512.0)
        for level, j in ((0.45, 40 + n), (0.8, 500 + n), (1.3, 1100 + n)):  # scores about 10, 18, 29
            k[j, 0] = level * unit
    got = ctx.run(q, k, v, host.Config(tokens, 1, 1, 512)).reshape(tokens, 1, 512)
    want = zo.attention_run(q, k, v, zo.Config(tokens, 1, 1, 512))
    refimpl.check_close(got, want, "rows overtaken several times")
    for n, i in enumerate(rows):
        assert np.abs(want[i, 0] - v[1100 + n, 0]).max() < 1e-2  # the last planted key takes the row


def test_wide_head_scores_that_outgrow_the_fixed_reference_are_formed_again(ctx):
    # The kernel exponentiates every score of a row against the largest score of the first
    # block of its key range; a workgroup whose row sums show a score more than 2^90 above that
    # flags its query tile and forms its rows of that range again with a running maximum.
    # Ordinary data flags nothing; a key 75 nats (108 in log2) above a field of N(0, 1)
    # scores, late in a range, flags its tile and only that one, and the rows still match.
    L = hip.lib()
    tokens = 1024
    rng = np.random.default_rng(79)
    q, k, v = draw(rng, tokens)
    cfg = host.Config(tokens, 1, 1, 512)
    got = ctx.run(q, k, v, cfg).reshape(tokens, 1, 512)
    assert L.zdraw_hip_wide_redo_tiles() == 0
    refimpl.check_close(got, zo.attention_run(q, k, v, zo.Config(tokens, 1, 1, 512)), "ordinary data")
    # rows 300 and 301 (tile 2) lean on keys 900 and 901, row 900 (tile 7) on key 1000: keys in the fifth and
    # the last block of the fourth key range (1024 tokens run as four ranges of eight blocks)
    for i, j in ((300, 900), (301, 901), (900, 1000)):
        k[j, 0] = 3.3 * q[i, 0] / np.linalg.norm(q[i, 0]) * np.sqrt(512.0)
    got = ctx.run(q, k, v, cfg).reshape(tokens, 1, 512)
    flagged = L.zdraw_hip_wide_redo_tiles()
    assert flagged == 2, flagged
    assert np.isfinite(got).all()
    want = zo.attention_run(q, k, v, zo.Config(tokens, 1, 1, 512))
    # (a bf16 operand's rounding error grows with the score: the planted rows are sharp one-hot
    # rows and are compared as such; every other row at the usual bar)
    others = np.ones(tokens, bool)
    others[[300, 301, 900]] = False
    refimpl.check_close(got[others], want[others], "rows beside the planted ones")
    for i, j in ((300, 900), (301, 901), (900, 1000)):
        assert np.abs(got[i, 0] - v[j, 0]).max() < 2e-2
    again = ctx.run(q, k, v, cfg).reshape(tokens, 1, 512)
    assert got.tobytes() == again.tobytes()


def rounded_reference(q, k, v):
    """Attention of one wide head in float64 on the operands the kernel multiplies: bf16, Q with its scale (exp2 domain)."""
    def bf16(x):
        return host.bf16_bits_to_f32(host.f32_to_bf16_bits(x)).reshape(x.shape)[:, 0].astype(np.float64)
    s = bf16(q * np.float32(np.log2(np.e) / np.sqrt(512.0))) @ bf16(k).T
    p = np.exp2(s - s.max(axis=1, keepdims=True))
    p /= p.sum(axis=1, keepdims=True)
    return p, (p @ bf16(v))[:, None]


# Rows formed again with a running maximum, over key ranges of any number of blocks: the loop there takes three
# blocks a trip, so 10, 7 and 4 blocks leave one over, 2 and 8 two, 9 none; ranges that end short (7, 4, 2); a row of a half-full last
# tile (its other waves have no row). Each row climbs twice: its first block is ordinary, a run of keys lies 108 (log2) above, which the
# fixed reference point cannot reach, and the last key another 9.5 above those, so that what has been summed is scaled by 2^-9.5
# once it counts: the run keeps a share of the row that shows, in the sum and in O. Operands rounded as the kernel rounds them:
# what is left is P and V in bf16, 2^-8 of the largest |V| (4.2) in all.
@pytest.mark.parametrize("tokens,part,blocks", [(64, 0, 2), (128, 0, 4), (256, 0, 8), (576, 1, 9), (640, 0, 10), (640, 1, 10), (1088, 3, 7), (1408, 5, 4), (1600, 6, 2)])
def test_wide_head_rows_formed_again_climb_twice(ctx, tokens, part, blocks):
    L = hip.lib()
    n, share = C.c_uint32(0), C.c_uint64(0)
    L.zdraw_hip_wide_ranges(tokens, 256, C.byref(n), C.byref(share))
    per = -(-(tokens // 32) // n.value)
    first = part * per
    assert part < n.value and min(per, tokens // 32 - first) == blocks, (n.value, per)
    rng = np.random.default_rng(80 + tokens + part)
    q, k, v = draw(rng, tokens)
    rows = (5, tokens - 1)
    last = 32 * (first + blocks) - 1
    run = {}
    for r, i in enumerate(rows):
        unit = q[i, 0] / np.linalg.norm(q[i, 0])
        per_bit = np.sqrt(512.0) / np.linalg.norm(q[i, 0]) / np.log2(np.e)  # |k| per unit of score (log2)
        run[i] = np.arange(32 * (first + 1) + r, last - 1, 2)  # every other key between the first block and the last two keys
        k[run[i], 0] = (108.0 * per_bit) * unit
        v[run[i], 0] = rng.standard_normal(512, dtype=np.float32)  # (one vector: their share is not averaged away)
        k[last - r, 0] = (117.5 * per_bit) * unit
    weight, want = rounded_reference(q, k, v)
    cfg = host.Config(tokens, 1, 1, 512)
    got = ctx.run(q, k, v, cfg).reshape(tokens, 1, 512)
    assert L.zdraw_hip_wide_redo_tiles() == len({i // 128 for i in rows})
    refimpl.check_close(got, want, f"{tokens} tokens, a range of {blocks} blocks formed again")
    for r, i in enumerate(rows):
        assert 0.015 < weight[i, run[i]].sum() < 0.5 and weight[i, last - r] > 0.5
    again = ctx.run(q, k, v, cfg).reshape(tokens, 1, 512)
    assert got.tobytes() == again.tobytes()


def test_wide_head_without_memory_for_the_shares_of_its_key_ranges(ctx):
    # the keys stay whole
    L = hip.lib()
    tokens = 3008
    n, share = C.c_uint32(), C.c_uint64()
    L.zdraw_hip_wide_ranges(tokens, 256, C.byref(n), C.byref(share))
    assert n.value > 1
    q, k, v = draw(np.random.default_rng(11), tokens)
    c2 = host.Context.init()  # a queue without scratch
    try:
        L.zdraw_hip_set_scratch_limit(tokens * 512 * 2)
        assert tokens * 512 * 2 < share.value
        got = c2.run(q, k, v, host.Config(tokens, 1, 1, 512)).reshape(tokens, 1, 512)
    finally:
        L.zdraw_hip_set_scratch_limit(0)
        c2.deinit()
    rows = [0, 127, tokens // 2, tokens - 65, tokens - 1]
    want = zo.attention_token_list(q, k, v, zo.Config(tokens, 1, 1, 512), rows)
    refimpl.check_close(got[rows], want.reshape(len(rows), 1, 512), "whole keys")
    ranges = ctx.run(q, k, v, host.Config(tokens, 1, 1, 512)).reshape(tokens, 1, 512)
    refimpl.check_close(got, ranges, "whole keys against key ranges")
    assert not np.array_equal(got, ranges)  # (the sums run in another order: it was the other form)


def test_wide_head_under_capture_does_not_grow_the_slot_of_its_shares(ctx):
    # a queue whose operand slots have room and whose share slot does not: the capture goes through with
    # whole keys, and every replay gives the bits of the call without memory for the shares
    L = hip.lib()
    tokens = 3008
    q, k, v = draw(np.random.default_rng(12), tokens)
    bufs = [ctx.buffer(a) for a in (q, k, v)] + [ctx.buffer(nbytes=q.nbytes)]
    err = C.create_string_buffer(128)
    wide = L.zdraw_hip_compile(ctx.device, None, b"attention_wide_mfma", err, 128)
    p = hip.AttnParams(tokens, 1, 1, 512, 0, 0)
    queue = L.zdraw_hip_create_queue(ctx.device)
    stream = C.c_void_p((C.c_void_p * 2).from_address(queue)[1])  # a queue is a device and a stream

    def enqueue(batch):
        return L.zdraw_hip_run_attention_enc_off(batch, wide, *(b.handle for b in bufs), C.byref(p), hip.K_WIDE, 512, 0, 0)

    batch = L.zdraw_hip_batch_begin(queue)
    try:
        L.zdraw_hip_set_scratch_limit(tokens * 512 * 2)
        assert enqueue(batch) == 0, hip.last_error()
        assert L.zdraw_hip_batch_end(batch) == 0
    finally:
        L.zdraw_hip_set_scratch_limit(0)
    want = bufs[3].read(np.uint32, q.shape)
    graph, run = C.c_void_p(), C.c_void_p()
    batch = L.zdraw_hip_batch_begin(queue)
    assert L.hipStreamBeginCapture(stream, C.c_int(2)) == 0
    rc = enqueue(batch)
    assert L.hipStreamEndCapture(stream, C.byref(graph)) == 0
    assert rc == 0, hip.last_error()
    assert L.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)) == 0
    for replay in range(3):
        bufs[3].write(np.full(q.nbytes, 0x7B, np.uint8))
        assert L.hipGraphLaunch(run, stream) == 0
        assert L.hipStreamSynchronize(stream) == 0
        assert np.array_equal(bufs[3].read(np.uint32, q.shape), want), f"replay {replay}"
    assert L.zdraw_hip_batch_end(batch) == 0
    assert L.hipGraphExecDestroy(run) == 0 and L.hipGraphDestroy(graph) == 0
    L.zdraw_hip_release_pipeline(wide)
    L.zdraw_hip_release_queue(queue)
    for b in bufs:
        b.release()


def test_wide_head_refusals_leave_nothing_enqueued(ctx):
    L = hip.lib()
    d0 = L.zdraw_hip_dispatch_count()
    z = np.zeros((96, 1, 512), np.float32)
    with pytest.raises(host.UnsupportedShape):  # tokens % 64 != 0 (mattn.zig:265)
        ctx.run(z, z, z, host.Config(96, 1, 1, 512))
    z2 = np.zeros((64, 2, 512), np.float32)
    with pytest.raises(host.UnsupportedShape):  # heads != 1 (mattn.zig:263)
        ctx.run(z2, z2, z2, host.Config(64, 2, 2, 512))
    z3 = np.zeros((64, 1, 256), np.float32)
    with pytest.raises(host.UnsupportedShape):
        ctx.run(z3, z3, z3, host.Config(64, 1, 1, 256))
    z4 = np.zeros((64, 1, 512), np.float32)
    with pytest.raises(host.UnsupportedShape):  # causal shapes are refused on the host
        ctx.run(z4, z4, z4, host.Config(64, 1, 1, 512, True))
    assert L.zdraw_hip_dispatch_count() == d0
    # C ABI: the wide pipeline runs kernel = wide only, and the block pipeline refuses width 512
    err = C.create_string_buffer(128)
    wide = L.zdraw_hip_compile(ctx.device, None, b"attention_wide_mfma", err, 128)
    assert wide, err.value
    assert L.zdraw_hip_pipeline_threads(wide) == 512
    b = ctx.buffer(z4)
    o = ctx.buffer(nbytes=z4.nbytes)
    p = hip.AttnParams(64, 1, 1, 512, 0, 0)
    assert L.zdraw_hip_run_attention(ctx.queue, wide, b.handle, b.handle, b.handle, o.handle, C.byref(p), hip.K_BLOCK, 512) == 1
    assert L.zdraw_hip_run_attention(ctx.queue, ctx.block_pipeline, b.handle, b.handle, b.handle, o.handle, C.byref(p), hip.K_BLOCK, 512) == 1
    p_short = hip.AttnParams(128, 1, 1, 512, 0, 0)  # buffers hold 64 rows
    assert L.zdraw_hip_run_attention(ctx.queue, wide, b.handle, b.handle, b.handle, o.handle, C.byref(p_short), hip.K_WIDE, 512) == 2
    assert L.zdraw_hip_dispatch_count() == d0
    assert L.zdraw_hip_run_attention(ctx.queue, wide, b.handle, b.handle, b.handle, o.handle, C.byref(p), hip.K_WIDE, 512) == 0
    assert L.zdraw_hip_dispatch_count() == d0 + 2  # rounding pass + attention
    # all-zero scores: every output row is the mean of V = 0
    assert not o.read(np.float32, z4.shape).any()
    L.zdraw_hip_release_pipeline(wide)
    b.release()
    o.release()


def test_wide_head_batch_offsets(ctx):
    # zdraw_metal_run_attention_enc_off: segments at byte offsets inside one buffer
    L = hip.lib()
    rng = np.random.default_rng(5)
    tokens, nseg = 128, 2
    q, k, v = (rng.standard_normal((nseg, tokens, 1, 512), dtype=np.float32) for _ in range(3))
    qb, kb, vb = ctx.buffer(q), ctx.buffer(k), ctx.buffer(v)
    ob = ctx.buffer(nbytes=q.nbytes)
    err = C.create_string_buffer(128)
    wide = L.zdraw_hip_compile(ctx.device, None, b"attention_wide_mfma", err, 128)
    p = hip.AttnParams(tokens, 1, 1, 512, 0, 0)
    seg = tokens * 512 * 4
    batch = L.zdraw_hip_batch_begin(ctx.queue)
    for i in range(nseg):
        assert L.zdraw_hip_run_attention_enc_off(batch, wide, qb.handle, kb.handle, vb.handle, ob.handle, C.byref(p),
                                                 hip.K_WIDE, 512, i * seg, i * seg) == 0, hip.last_error()
    assert L.zdraw_hip_batch_end(batch) == 0
    got = ob.read(np.float32, q.shape)
    for i in range(nseg):
        refimpl.check_close(got[i], zo.attention_run(q[i], k[i], v[i], zo.Config(tokens, 1, 1, 512)), f"segment {i}")
    L.zdraw_hip_release_pipeline(wide)
    for b in (qb, kb, vb, ob):
        b.release()
