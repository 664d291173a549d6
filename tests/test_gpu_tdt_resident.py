"""The resident TDT decode (weights in LDS, every window of a launch sharing
them) against the decode with one workgroup per window: bit-identical
tokens, states and scratch at the edges of its launch shapes, with head
weights that are not finite, on two streams at once, and when its workgroups,
or those and the teams behind them, give up waiting."""
import numpy as np
import pytest

from test_gpu_encoder import Stack
from test_gpu_parity import Scope

pytestmark = pytest.mark.gpu

OUTPUTS = ("tokens", "token_frames", "token_durations", "metadata", "state", "predictor_scratch")


@pytest.fixture
def scope(ctx):
    s = Scope(ctx)
    yield s
    s.close()


class Decoder:
    def __init__(self, abi, scope, ctx, case, precision, max_tokens=512):
        B = case.batch
        fill = np.full((B, max_tokens), 0xDEADBEEF, np.uint32)
        self.out = {n: scope.put(fill) for n in OUTPUTS[:3]}
        self.out["metadata"] = scope.put(np.full(2 * B, 0xDEADBEEF, np.uint32))
        self.out["state"] = scope.put(np.full((B, 4, 640), 3.0, np.float32))
        self.out["predictor_scratch"] = scope.put(np.full((B, 5, 640), 5.0, np.float32))
        self.op = abi.TdtDecoderOp(ctx, weights={k: scope.put(case.weights[k]) for k in abi.TDT_WEIGHT_NAMES},
                                   encoder_projected=scope.put(case.encoder_projected),
                                   encoded_lengths=scope.put(case.lengths), decode_starts=scope.put(case.starts),
                                   decode_ends=scope.put(case.ends), flush_finals=scope.put(case.flush),
                                   batch_size=B, frames=case.frames, max_tokens=max_tokens, precision=precision,
                                   **self.out)

    def words(self):
        return {n: b.download().view(np.uint32) for n, b in self.out.items()}


def decode(abi, scope, ctx, case, precision, *, team=None, polls=None, join=None, team_polls=None, active=0):
    d = Decoder(abi, scope, ctx, case, precision)
    try:
        if team is not None:
            d.op.set_team_size(team)
        assert bool(d.op.resident_windows()) == (team is None)
        if polls is not None:
            d.op.set_wait_limit(polls)
        if join is not None:
            d.op.set_join_limit(join)
        if team_polls is not None:
            d.op.set_team_limit(team_polls)
        print(precision, "batch", case.batch, "team", team, "polls", polls, "join", join, flush=True)
        assert d.op.abandoned_launches() == 0
        d.op.enqueue(active)
        ctx.synchronize()
        given_up = polls is not None or join is not None
        launches = -(-(active or case.batch) // d.op.resident_windows()) if given_up else 0
        assert d.op.abandoned_launches() == launches
        return d.words()
    finally:
        d.op.release()


def same(got, want):
    for name in OUTPUTS:
        np.testing.assert_array_equal(got[name], want[name], err_msg=name)


def ragged(workloads, seed, batch, precision, blank_bias, frames=40):
    """Full, one-frame, empty and bounded windows, the flush on every other."""
    rng = np.random.default_rng(seed)
    lengths = rng.integers(frames // 2, frames + 1, batch)
    lengths[::5], lengths[1::7] = frames, 1
    starts, ends = np.zeros(batch, int), np.full(batch, frames)
    if batch > 3:
        lengths[3] = 0
        starts[2], ends[2] = 3, frames - 5
    return workloads.tdt_case(seed, batch, frames, lengths=lengths, starts=starts, ends=ends,
                              flush=np.arange(batch) % 2, blank_bias=blank_bias, precision=precision)


# one and more windows per wave, their partial waves, one and more launches
@pytest.mark.parametrize("precision,batch", [("f16", b) for b in (1, 2, 4, 5, 7, 9, 16, 17, 33, 64)] +
                         [("f32", b) for b in (1, 3, 4, 5, 6, 7, 24)])
def test_resident_decode_matches_one_workgroup_per_window(abi, ctx, scope, workloads, precision, batch):
    case = ragged(workloads, 20 + batch, batch, precision, 1.0)
    same(decode(abi, scope, ctx, case, precision), decode(abi, scope, ctx, case, precision, team=1))


@pytest.mark.parametrize("precision", ["f16", "f32"])
def test_resident_decode_leaves_out_zero_inputs_of_weights_that_are_not_finite(abi, ctx, scope, workloads, precision):
    case = ragged(workloads, 5, 5, precision, 1.0)
    head = case.weights["head_weight"]
    head[11, 3], head[200, 1026], head[639, 1000] = np.inf, -np.inf, np.nan
    case.weights["head_bias"][[5, 9]] = np.nan, -np.inf
    same(decode(abi, scope, ctx, case, precision), decode(abi, scope, ctx, case, precision, team=1))


@pytest.mark.parametrize("team_polls", [None, 0])  # the teams behind it decode, or give up as well
@pytest.mark.parametrize("limit", ["polls", "join"])
@pytest.mark.parametrize("precision,batch", [("f16", 3), ("f16", 33), ("f32", 7)])
def test_resident_decode_that_gives_up_is_decoded_again(abi, ctx, scope, workloads, precision, batch, limit,
                                                                team_polls):
    case = ragged(workloads, 40 + batch, batch, precision, 0.5)
    same(decode(abi, scope, ctx, case, precision, team_polls=team_polls, **{limit: 0}),
         decode(abi, scope, ctx, case, precision, team=1))


def test_resident_decodes_on_two_streams_and_an_active_prefix(abi, ctx, scope, workloads):
    """Two ops enqueued on two streams without a synchronisation between
    them; then a prefix, which leaves the other windows' outputs alone."""
    cases = [ragged(workloads, 60 + i, 9, p, 0.5) for i, p in enumerate(("f16", "f32"))]
    want = [decode(abi, scope, ctx, c, p, team=1) for c, p in zip(cases, ("f16", "f32"))]
    other = abi.ctypes.c_void_p()
    abi.check(abi.load().pk_stream_create(ctx.handle, abi.ctypes.byref(other)))
    ops = [Decoder(abi, scope, ctx, c, p) for c, p in zip(cases, ("f16", "f32"))]
    try:
        ctx.synchronize()
        for _ in range(3):
            for d, stream in zip(ops, (None, other)):
                d.op.enqueue(0, stream)
        ctx.synchronize()
        ctx.synchronize(other)
        for d, w in zip(ops, want):
            assert d.op.abandoned_launches() == 0
            same(d.words(), w)
    finally:
        for d in ops:
            d.op.release()
        abi.check(abi.load().pk_stream_destroy(ctx.handle, other))
    same(decode(abi, scope, ctx, cases[0], "f16", active=5), decode(abi, scope, ctx, cases[0], "f16", team=1, active=5))


@pytest.mark.parametrize("precision", ["f16", "f32"])
def test_resident_decode_beside_encoder_passes(abi, ctx, scope, workloads, precision):
    """Decodes on one stream while encoder passes run on another: both as when
    alone, to the bit, and no launch is given up for the passes' sake."""
    case = ragged(workloads, 80, 6, precision, 0.5)
    want = decode(abi, scope, ctx, case, precision, team=1)
    encoder = Stack(abi, ctx, scope, workloads.encoder_stack(seed=81, windows=8, frames=188, layers=2))
    decoder = Decoder(abi, scope, ctx, case, precision)
    other = abi.ctypes.c_void_p()
    abi.check(abi.load().pk_stream_create(ctx.handle, abi.ctypes.byref(other)))
    try:
        alone = encoder.run(graph=True)
        for _ in range(4):
            encoder.op.enqueue(graph=True)
            decoder.op.enqueue(0, other)
            encoder.op.enqueue(graph=True)
        ctx.synchronize()
        ctx.synchronize(other)
        assert decoder.op.abandoned_launches() == 0
        same(decoder.words(), want)
        np.testing.assert_array_equal(encoder.output.download().view(np.uint16), alone.view(np.uint16))
    finally:
        decoder.op.release()
        encoder.release()
        abi.check(abi.load().pk_stream_destroy(ctx.handle, other))
