"""The affine u8 stores: single tokens coded by the attention launch, prompts in chunks of every length, prompt buffers that are
handed out again.  Stored bytes and parameters against the oracle, bit for bit."""
import ctypes as C

import numpy as np
import pytest

import tract_amd
from oracle import oracle as orc
from tests.gpu_util import rt  # noqa: F401
from tract_amd import _lib, kivi
from tract_amd._lib import call
from tract_amd.runtime import Stream

pytestmark = pytest.mark.gpu
D = 128


def _same(got, want):
    assert got["packed"].tobytes() == want["packed"].tobytes()
    assert got["lo"].tobytes() == want["lo"].tobytes() and got["scale"].tobytes() == want["scale"].tobytes()


# from the first token on, across tiles of 32 and the four waves of a workgroup; 4, 8 and 16 heads per kv head (records of 8 and
# of 16 rows); minima and ranges that move late, constant rows, a range of exactly zero
@pytest.mark.parametrize("B,Hq,Hkv,steps", [(1, 8, 2, 140), (2, 16, 2, 70), (1, 16, 1, 40)])
def test_single_tokens_from_an_empty_store(rt, B, Hq, Hkv, steps):
    rng = np.random.default_rng(steps)
    st = tract_amd.QuantizedKvSdpa(axis=2).state()
    kc, vc = orc.KiviCache(True, running=True), orc.KiviCache(False, running=True)
    for t in range(steps):
        q = (rng.standard_normal((B, Hq, 1, D)) / np.sqrt(D)).astype(np.float16)
        k, v = rng.standard_normal((B, Hkv, 1, D)).astype(np.float16), rng.standard_normal((B, Hkv, 1, D)).astype(np.float16)
        k[:, :, :, 3] *= np.float16(1 + 8 * t)      # ranges beyond 255: the scale moves with every token
        k[:, :, :, 4] = np.float16(-t)
        if t % 9 == 4:
            v[:] = np.float16(-3.25)
        got = st.eval([q, k, v]).to_numpy().astype(np.float64)
        kc.ingest(k.astype(np.float32)), vc.ingest(v.astype(np.float32))
        if t < 3 or t % 31 == 0 or t == steps - 1:
            want = orc.flash_sdpa(q.astype(np.float32), kc.dequantized(), vc.dequantized(), causal=False)
            assert np.abs(got - want).max() <= 2e-2, t   # (the tolerance of the existing step tests: f16 products over a sharp softmax)
            _same(st.k.state(), kc.state()), _same(st.v.state(), vc.state())


# chunks of 8, 16, 32 and 64 tokens, one token more and less than each change, on top of earlier state
@pytest.mark.parametrize("lengths", [(63, 64, 65), (512, 5, 513), (4096, 1), (4097, 70), (8193,)])
def test_prompts_in_chunks_of_every_length(rt, lengths):
    rng = np.random.default_rng(lengths[0])
    cache = kivi.KiviCache(kivi.KIVI_RUNNING_CHANNEL, 8, 0, 1, 2, D)
    ref = orc.KiviCache(True, running=True)
    for n in lengths:
        x = (rng.standard_normal((1, 2, n, D)) * 100).astype(np.float16)
        x[0, 1, :, 9] = np.linspace(5, -600, n).astype(np.float16)
        x[0, 0, n // 2, 3] = np.nan
        cache.append(x)
        ref.ingest(x.astype(np.float32))
        _same(cache.state(), ref.state())


def test_sessions_that_reuse_their_prompt_buffers(rt):
    """Prompt, steps, reset, again, on two streams in turn without a wait in between: the buffers a prompt left behind serve a
    later one, and every session gives what it gave alone."""
    rng = np.random.default_rng(3)
    data = []
    for n in (300, 200, 260):
        data.append([((rng.standard_normal((1, 8, m, D)) / np.sqrt(D)).astype(np.float16), rng.standard_normal((1, 2, m, D)).astype(np.float16),
                      rng.standard_normal((1, 2, m, D)).astype(np.float16)) for m in (n, 1, 1)])
    alone = []
    for calls in data:
        st = tract_amd.QuantizedKvSdpa(axis=2).state()
        alone.append([st.eval(list(c)).to_numpy() for c in calls])
    streams = [Stream(), Stream()]
    states = [tract_amd.QuantizedKvSdpa(axis=2).state() for _ in streams]
    device = [[[tract_amd.DeviceTensor.from_numpy(t) for t in c] for c in calls] for calls in data]
    outs = []
    for turn in range(6):
        i, calls = turn % 3, device[turn % 3]
        st, s = states[turn % 2], streams[turn % 2]
        if st.k is not None:
            st.k.reset(stream=s), st.v.reset(stream=s)
        outs.append((i, s, [st.eval(c, stream=s) for c in calls]))
    for i, s, got in outs:
        for g, w in zip(got, alone[i]):
            assert np.array_equal(g.to_numpy(s), w)


# rows that start one and two elements past an aligned address: the same bits, and the step that needs no dequantised copy
@pytest.mark.parametrize("off_k,off_v", [(1, 0), (0, 1), (2, 3), (1, 1)])
def test_single_tokens_at_any_element(rt, off_k, off_v):
    rng = np.random.default_rng(off_k + 10 * off_v)
    B, Hq, Hkv = 2, 8, 2
    data = [((rng.standard_normal((B, Hq, n, D)) / np.sqrt(D)).astype(np.float16), rng.standard_normal((B, Hkv, n, D)).astype(np.float16),
             rng.standard_normal((B, Hkv, n, D)).astype(np.float16)) for n in (40, 1, 1, 1)]

    def shifted(x, off):
        t = tract_amd.DeviceTensor.from_numpy(np.concatenate([np.zeros(off, np.float16), x.reshape(-1)]))
        return tract_amd.DeviceTensor(x.shape, np.float16, ptr=t.ptr.value + 2 * off, owner=t)

    aligned, moved = tract_amd.QuantizedKvSdpa(axis=2).state(), tract_amd.QuantizedKvSdpa(axis=2).state()
    for q, k, v in data:
        step = k.shape[2] == 1
        want = aligned.eval([q, k, v]).to_numpy()
        got = moved.eval([tract_amd.DeviceTensor.from_numpy(q), shifted(k, off_k) if step else k, shifted(v, off_v) if step else v]).to_numpy()
        np.testing.assert_array_equal(got, want)
        _same(moved.k.state(), aligned.k.state()), _same(moved.v.state(), aligned.v.state())


def test_a_recorded_step_replayed_in_later_sessions(rt):
    """A step recorded into a graph, replayed after other prompts of the same length with numbers of single tokens in between
    that are odd and even: every replay gives what the step gives in a new session."""
    rng = np.random.default_rng(17)
    B, Hq, Hkv, n = 2, 8, 2, 41

    def tokens(m, scale=1.0):
        return [(rng.standard_normal((B, h, m, D)) * s).astype(np.float16) for h, s in ((Hq, D ** -0.5), (Hkv, scale), (Hkv, scale))]

    def eager(calls):
        st = tract_amd.QuantizedKvSdpa(axis=2).state()
        return [st.eval(c).to_numpy() for c in calls][-1]

    hip, s, held = _lib.load(), Stream(), [tract_amd.DeviceTensor.from_numpy(t) for t in tokens(1)]
    out = tract_amd.DeviceTensor((B, Hq, 1, D), np.float16)
    st = tract_amd.QuantizedKvSdpa(axis=2).state()

    def put(step):
        for t, x in zip(held, step):
            call("trocm_h2d", t.ptr, x.ctypes.data_as(C.c_void_p), t.nbytes, s.handle)
            s.synchronize()

    def check(rc):
        assert rc == 0, rc

    def on_device(step):
        return [tract_amd.DeviceTensor.from_numpy(t, s) for t in step]

    graph, runnable = C.c_void_p(), C.c_void_p()
    for session, more in enumerate((0, 1, 2, 3)):
        scale = 4.0 ** -session   # (ranges of an earlier session would give other codes)
        prompt, first, step = tokens(n, scale), tokens(1, scale), tokens(1, scale)
        if session:
            for _ in range(more):
                st.eval(on_device(tokens(1, 30.0)), stream=s)
            st.k.reset(stream=s), st.v.reset(stream=s)
        for c in (prompt, first):
            st.eval(on_device(c), stream=s)
        put(step)
        if session == 0:
            check(hip.hipStreamBeginCapture(s.handle, 2))
            st.eval(held, stream=s, out=out)
            check(hip.hipStreamEndCapture(s.handle, C.byref(graph)))
            check(hip.hipGraphInstantiate(C.byref(runnable), graph, None, None, C.c_size_t(0)))
        for _ in range(2):   # (the same token again: the same row and parameters)
            check(hip.hipGraphLaunch(runnable, s.handle))
            np.testing.assert_array_equal(out.to_numpy(s), eager([prompt, first, step]))
    check(hip.hipGraphExecDestroy(runnable))
    check(hip.hipGraphDestroy(graph))


@pytest.mark.parametrize("over", ["k", "v"])
def test_a_step_stored_over_its_own_new_rows(rt, over):
    """More workgroups than run at once, so that some read their rows after others have stored results."""
    rng = np.random.default_rng(23)
    B, Hq, Hkv = 192, 32, 8
    data = [tuple((rng.standard_normal((B, h, n, D)) * c).astype(np.float16) for h, c in ((Hq, D ** -0.5), (Hkv, 1), (Hkv, 1))) for n in (33, 1, 1)]
    apart, shared = tract_amd.QuantizedKvSdpa(axis=2).state(), tract_amd.QuantizedKvSdpa(axis=2).state()
    for q, k, v in data:
        want = apart.eval([q, k, v]).to_numpy()
        args = {name: tract_amd.DeviceTensor.from_numpy(t) for name, t in (("q", q), ("k", k), ("v", v))}
        out = tract_amd.DeviceTensor(q.shape, np.float16)
        if k.shape[2] == 1:
            whole = np.zeros(q.size, np.float16)
            whole[: k.size] = (k if over == "k" else v).reshape(-1)
            out = tract_amd.DeviceTensor.from_numpy(whole.reshape(q.shape))
            args[over] = tract_amd.DeviceTensor(k.shape, np.float16, ptr=out.ptr, owner=out)
        np.testing.assert_array_equal(shared.eval([args["q"], args["k"], args["v"]], out=out).to_numpy(), want)
        _same(shared.k.state(), apart.k.state()), _same(shared.v.state(), apart.v.state())


def test_a_recorded_prompt_keeps_its_copies(rt):
    """A prompt and a step recorded together: the step hands the prompt's dequantised copies back, and they stay the graph's
    whatever is released or allocated between its replays."""
    rng = np.random.default_rng(29)
    B, Hq, Hkv, n = 1, 8, 2, 70

    def tokens(m):
        return [(rng.standard_normal((B, h, m, D)) * c).astype(np.float16) for h, c in ((Hq, D ** -0.5), (Hkv, 1), (Hkv, 1))]

    hip, s = _lib.load(), Stream()
    calls = [tokens(n), tokens(1)]
    alone = tract_amd.QuantizedKvSdpa(axis=2).state()
    want = [alone.eval(c).to_numpy() for c in calls]
    held = [[tract_amd.DeviceTensor.from_numpy(t) for t in c] for c in calls]
    outs = [tract_amd.DeviceTensor(c[0].shape, np.float16) for c in calls]
    st = tract_amd.QuantizedKvSdpa(axis=2).state()
    for c in calls:   # (rows, workspace and scratch are there; the copies go to the list and are released)
        st.eval([tract_amd.DeviceTensor.from_numpy(t) for t in c], stream=s)
    s.synchronize()
    call("trocm_release_unused", 1)
    st.k.reset(stream=s), st.v.reset(stream=s)
    s.synchronize()
    graph, runnable = C.c_void_p(), C.c_void_p()
    assert hip.hipStreamBeginCapture(s.handle, 2) == 0
    for c, out in zip(held, outs):
        st.eval(c, stream=s, out=out)
    assert hip.hipStreamEndCapture(s.handle, C.byref(graph)) == 0
    assert hip.hipGraphInstantiate(C.byref(runnable), graph, None, None, C.c_size_t(0)) == 0
    others = []
    for _ in range(3):
        others.append(tract_amd.QuantizedKvSdpa(axis=2).state())
        for c, w in zip(calls, want):
            np.testing.assert_array_equal(others[-1].eval([tract_amd.DeviceTensor.from_numpy(t) for t in c], stream=s).to_numpy(s), w)
        call("trocm_release_unused", 1)
        st.k.reset(stream=s), st.v.reset(stream=s)   # (a replay is a session from the start)
        assert hip.hipGraphLaunch(runnable, s.handle) == 0
        for out, w in zip(outs, want):
            np.testing.assert_array_equal(out.to_numpy(s), w)
    assert hip.hipGraphExecDestroy(runnable) == 0
    assert hip.hipGraphDestroy(graph) == 0
