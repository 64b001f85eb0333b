"""Parity of the HIP dense decode (benchmark config 4's structure) with the oracle on an MI355X,
through the C ABI (the persistent run, lxm_dn_run, the per-step kernels, lxm_dn_step, and the
batched prefill, lxm_dn_prefill, followed by steps): predictions and final states bit for bit. The dense projections are summed in
the dense order the oracle restates for matrices marked dense (64 groups of a row's entries in
order from +0, then the pairwise tree); everything else follows the stock decode as in the
sparse paths. Sizes: config 4's layout scaled down (hidden 256, 2 layers) so the oracle runs in
seconds; the full config is measured by bench.py (--legs dense).
"""

import numpy as np
import pytest
import torch

from linuxformer_amd import chunk, dense, fast, mk_build, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def cuda():
    assert torch.cuda.is_available(), "the gpu tests need an MI355X"
    mk_build.load()
    return torch.device("cuda", 0)


_M = {}


def model(name="small"):
    if name not in _M:
        spec = synth.config4_small() if name == "small" else synth.config4_mid()
        dm_cpu = synth.build_dense(spec, "cpu")
        _M[name] = (spec, dm_cpu, synth.to_sparse(dm_cpu))
    return _M[name]


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


def check(n_forced, n, seed=None, graph=True, name="small", mode="persistent"):
    from oracle import oracle as ox

    spec, dm_cpu, sm = model(name)
    conv0, rec0 = synth.dense_state(dm_cpu, seed)
    forced = [int(x) for x in np.random.default_rng(7 + n_forced).integers(0, spec.vocab, n_forced)]
    print(f"[gpu-test] dense {spec.name}: forced={n_forced} n={n} seed={seed} mode={mode} "
          f"graph={graph}", flush=True)
    dm = synth.dense_to(dm_cpu, "cuda")
    cache = fast.StateCache(conv0, rec0, "bf16", "cuda")
    dd = dense.DenseDecode(dm, cache)
    preds = dd.run(forced, n, graph=graph, mode=mode)
    c, r = conv0.copy(), rec0.copy()
    po, _, _ = ox.OracleModel(sm).decode(c, r, forced, n)
    assert preds == po.tolist()
    assert (bits(cache.conv_numpy()) == bits(c)).all()
    assert (bits(cache.rec_numpy()) == bits(r)).all()
    return preds


MODES = ["persistent", "steps"]


@pytest.mark.parametrize("mode", MODES)
def test_dense_small_greedy(cuda, mode):
    check(1, 24, mode=mode)


@pytest.mark.parametrize("mode", MODES)
def test_dense_small_forced_then_greedy(cuda, mode):
    """A forced prefix (the config's prefill, scaled down), then greedy steps."""
    check(16, 32, mode=mode)


def test_dense_small_live_state_eager(cuda):
    """From N(0, 1) states and nonzero windows on the live heads, eager steps (no graph)."""
    check(4, 12, seed=3, graph=False, mode="steps")


def test_dense_small_live_state_graph(cuda):
    check(4, 12, seed=3, graph=True, mode="steps")


def test_dense_persistent_phase_clock(cuda):
    """The profiling build's persistent run (its phase clock on) predicts what the oracle does and
    fills the clock: every workgroup's six phases, each use counted in ticks."""
    from oracle import oracle as ox

    spec, dm_cpu, sm = model("small")
    conv0, rec0 = synth.dense_state(dm_cpu, 3)
    forced = [int(x) for x in np.random.default_rng(11).integers(0, spec.vocab, 3)]
    print(f"[gpu-test] dense {spec.name}: persistent run with the phase clock", flush=True)
    dm = synth.dense_to(dm_cpu, "cuda")
    cache = fast.StateCache(conv0, rec0, "bf16", "cuda")
    dd = dense.DenseDecode(dm, cache, subprof=True)
    ncu = torch.cuda.get_device_properties(0).multi_processor_count
    prof = torch.zeros(32 * ncu, dtype=torch.int64, device="cuda")
    preds = dd.run(forced, 10, mode="persistent", prof=prof)
    c, r = conv0.copy(), rec0.copy()
    po, _, _ = ox.OracleModel(sm).decode(c, r, forced, 10)
    assert preds == po.tolist()
    assert (bits(cache.rec_numpy()) == bits(r)).all()
    acc = prof.view(ncu, 32)[:, :18].cpu().numpy().reshape(ncu, 6, 3)
    assert (acc[:, :, 1:].sum(axis=2) > 0).all()  # every phase's rows and barrier took time
    assert (acc >= 0).all() and (acc[:, 5, 1] > 0).all()  # the head's rows on every workgroup
    with pytest.raises(ValueError):
        dd.run(forced, 2, mode="persistent", prof=prof[:16])


def test_dense_small_live_state_persistent(cuda):
    check(4, 12, seed=3)


@pytest.mark.parametrize("mode", MODES)
def test_dense_full_widths(cuda, mode):
    """Config 4's full row lengths (hidden 2560: 40 entries per lane; SwiGLU 9216: 144; 16 key
    heads x 2 live value heads: 4096 out_proj entries, 64) over one layer, from live states."""
    check(3, 6, seed=5, name="mid", mode=mode)


def check_prefill(T, n, seed=None, name="small"):
    """lxm_dn_prefill over T - 1 forced tokens, then n steps from the last one: the predictions
    and states of T - 1 + n steps of the oracle with the same T forced tokens."""
    from oracle import oracle as ox

    spec, dm_cpu, sm = model(name)
    conv0, rec0 = synth.dense_state(dm_cpu, seed)
    toks = [int(x) for x in np.random.default_rng(11 + T).integers(0, spec.vocab, T)]
    print(f"[gpu-test] dense prefill {spec.name}: T={T} n={n} seed={seed}", flush=True)
    dm = synth.dense_to(dm_cpu, "cuda")
    cache = fast.StateCache(conv0, rec0, "bf16", "cuda")
    dd = dense.DenseDecode(dm, cache)
    dd.prefill(toks[:-1])
    preds = dd.run(toks[-1:], n)
    c, r = conv0.copy(), rec0.copy()
    po, _, _ = ox.OracleModel(sm).decode(c, r, toks, T - 1 + n)
    assert preds == po.tolist()[T - 1:]
    assert (bits(cache.conv_numpy()) == bits(c)).all()
    assert (bits(cache.rec_numpy()) == bits(r)).all()


@pytest.mark.parametrize("T,seed", [(40, None), (3, 3), (34, 3)])
def test_dense_prefill_small(cuda, T, seed):
    """Batches of 16 (the last one partial), a prompt shorter than the conv window, live states."""
    check_prefill(T, 6, seed=seed)


@pytest.mark.parametrize("n", [1, 16, 17, 32, 33, 64, 65, 97])
def test_dense_prefill_token_tiles(cuda, n):
    """Prompts at the row kernels' token tiles (16, 32 or 64 tokens on 16-row tiles, 64 a workgroup
    on 32-row tiles beyond): whole tiles, one past them, one token alone."""
    check_prefill(n + 1, 2, seed=3)


@pytest.mark.parametrize("kl,zeros", [(128, True), (160, False), (160, True), (256, False)])
def test_dense_prefill_key_dims(cuda, kl, zeros):
    """The delta rule's forms: 8 row blocks up to 128 live key dims and 16 beyond; tokens whose query
    and key hold zeros among the live dims (a third of the query/key rows zero) and a key head that
    is all zero, beside tokens with none."""
    from dataclasses import replace

    from oracle import oracle as ox

    spec = replace(synth.config4_small(), kd_live=kl)
    dm = synth.build_dense(spec, "cpu")
    conv0, rec0 = synth.dense_state(dm, 3)
    if zeros:
        for ly in dm.layers:
            ly["qk"][:, :, ::3] = 0
            ly["qk"][:, 1] = 0
    conv0[:, :2 * spec.nk * 256] = 0.0
    toks = [int(x) for x in np.random.default_rng(17).integers(0, spec.vocab, 21)]
    print(f"[gpu-test] dense prefill key dims: kl={kl} zeros={zeros}", flush=True)
    cache = fast.StateCache(conv0, rec0, "bf16", "cuda")
    dense.DenseDecode(synth.dense_to(dm, "cuda"), cache).prefill(toks)
    c, r = conv0.copy(), rec0.copy()
    ox.OracleModel(synth.to_sparse(dm)).decode(c, r, toks, len(toks))
    assert (bits(cache.conv_numpy()) == bits(c)).all()
    assert (bits(cache.rec_numpy()) == bits(r)).all()


@pytest.mark.parametrize("kl", [64, 128, 160])
@pytest.mark.parametrize("kind", ["key", "decay", "value", "large"])
def test_dense_prefill_not_finite(cuda, kl, kind):
    """Weights that make a key, a decay or a value NaN or infinite, and products that overflow: the live
    heads' states and windows are NaN where the oracle's are (a NaN key or decay reaches the zero rows
    past the live key dims, a value only its column) and its bits elsewhere."""
    from dataclasses import replace

    from oracle import oracle as ox

    spec = replace(synth.config4_small(), kd_live=kl)
    dm = synth.build_dense(spec, "cpu")
    conv0, rec0 = synth.dense_state(dm, 3)
    ly = dm.layers[0]
    if kind == "key":
        ly["qk"][1, 1, 3, 5] = float("nan")
    elif kind == "decay":
        ly["a"][0, 1, 7] = float("nan")
    elif kind == "value":
        ly["v"][0, 0, 3, 5] = float("inf")
    else:
        for ly in dm.layers:
            for n in ("qk", "v", "z", "b", "a", "out", "gate", "up", "down"):
                ly[n] = (ly[n].float() * 1e30).bfloat16()
    toks = [int(x) for x in np.random.default_rng(29).integers(0, spec.vocab, 21)]
    print(f"[gpu-test] dense prefill not finite: kl={kl} {kind}", flush=True)
    cache = fast.StateCache(conv0, rec0, "bf16", "cuda")
    dense.DenseDecode(synth.dense_to(dm, "cuda"), cache).prefill(toks)
    c, r = conv0.copy(), rec0.copy()
    ox.OracleModel(synth.to_sparse(dm)).decode(c, r, toks, len(toks))
    # (the dead heads and channels: the kernels leave them alone, the oracle's 0 x NaN does not)
    R = spec.nv // spec.nk

    def live(conv, rec):
        rec = rec.reshape(-1, spec.nk, R, 256, 128)[:, :, :spec.r_live]
        nq = 2 * spec.nk * 256
        qk = conv[:, :nq].reshape(-1, 2 * spec.nk, 256, 4)[:, :, :kl]
        return rec, qk, conv[:, nq:].reshape(-1, spec.nk, R, 128, 4)[:, :, :spec.r_live]

    got, want = live(cache.conv_numpy(), cache.rec_numpy()), live(c, r)
    assert any(np.isnan(w).any() for w in want)
    for x, y in zip(got, want):
        assert (np.isnan(x) == np.isnan(y)).all()
        assert (bits(x)[~np.isnan(y)] == bits(y)[~np.isnan(y)]).all()


@pytest.mark.parametrize("n", [5, 40])
def test_dense_prefill_repeats(cuda, n):
    """The same prompt twice leaves the same bits at the full row lengths (a short prompt's kernels
    keep many workgroups a CU, whose waves drift apart: a stage written before every wave has read
    it shows as a difference between runs)."""
    spec, dm_cpu, _ = model("mid")
    dm = synth.dense_to(dm_cpu, "cuda")
    conv0, rec0 = synth.dense_state(dm_cpu, 3)
    toks = [int(x) for x in np.random.default_rng(n).integers(0, spec.vocab, n)]
    print(f"[gpu-test] dense prefill repeats: n={n}", flush=True)
    out = []
    for _ in range(6):
        cache = fast.StateCache(conv0, rec0, "bf16", "cuda")
        dense.DenseDecode(dm, cache).prefill(toks)
        out.append((cache.conv_numpy(), cache.rec_numpy()))
    for a in out[1:]:
        assert (bits(a[0]) == bits(out[0][0])).all() and (bits(a[1]) == bits(out[0][1])).all()


@pytest.mark.parametrize("chunked,nt", [(0, 16), (0, 48), (1, 64), (1, 128)])
def test_dense_prefill_batches(cuda, chunked, nt):
    """The C entries with buffers of nt tokens (16 and 64: lxm_dn_prefill and
    lxm_dn_prefill_chunked; other sizes: lxm_dn_prefill_n) leave the same bits as one batch of the
    whole prompt: 150 tokens, so that every size has a partial last batch."""
    import ctypes

    spec, dm_cpu, _ = model()
    conv0, rec0 = synth.dense_state(dm_cpu, 3)
    toks = [int(x) for x in np.random.default_rng(31).integers(0, spec.vocab, 150)]
    print(f"[gpu-test] dense prefill batches: chunked={chunked} nt={nt}", flush=True)
    dm = synth.dense_to(dm_cpu, "cuda")
    out = []
    for whole in (True, False):
        cache = fast.StateCache(conv0, rec0, "bf16", "cuda")
        dd = dense.DenseDecode(dm, cache)
        if whole:
            dd.prefill(toks, mode="chunked" if chunked else "batched")
        else:
            pb, _ = dd._pbuf(nt)
            tok = torch.tensor(toks, dtype=torch.int32, device="cuda")
            p, _ = dd._params(1)
            args = [ctypes.byref(p), ctypes.c_void_p(tok.data_ptr()), len(toks), ctypes.byref(pb)]
            st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
            if nt == 16:
                e = dd.lib.lxm_dn_prefill(*args, st)
            elif nt == 64:
                e = dd.lib.lxm_dn_prefill_chunked(*args, st)
            else:
                ws = chunk.workspace(spec.nk * spec.r_live, 64, "cuda")  # (one chunk a group)
                e = dd.lib.lxm_dn_prefill_n(*args, nt, chunked, ctypes.c_void_p(ws.data_ptr()),
                                            ws.numel(), st)
            assert e == 0
            torch.cuda.synchronize()
        out.append((cache.conv_numpy(), cache.rec_numpy()))
    for a, b in zip(*out):
        assert (bits(a) == bits(b)).all()


def fma_chain(a, b):
    """sum_k a[:, k] b[:, k]' from +0 in k order, each step one fused multiply-add rounded to the nearest
    even float32, denormals kept: products of float32 are exact in float64; the sum is rounded to odd
    there (53 bits), so the rounding to 24 is the only one."""
    acc = np.zeros((a.shape[0], b.shape[0]), np.float32)
    for k in range(a.shape[1]):
        p = a[:, k].astype(np.float64)[:, None] * b[:, k].astype(np.float64)[None]
        c = acc.astype(np.float64)
        s = c + p
        t = s - c
        e = (c - (s - t)) + (p - t)
        odd = np.isfinite(s) & np.isfinite(e) & (e != 0) & (s.view(np.uint64) & 1 == 0)
        s = np.where(odd, np.nextafter(s, np.where(e > 0, np.inf, -np.inf)), s)
        acc = s.astype(np.float32)
    return acc


REGIMES = ["normal", "wide", "cancel", "denormal_in", "denormal_out", "overflow", "not_finite",
           "float32"]


@pytest.mark.parametrize("rows", [32, 16])
@pytest.mark.parametrize("regime", REGIMES)
@np.errstate(all="ignore")
def test_mfma_sums_are_fma_chains(cuda, rows, regime):
    """What the prompt's row kernels rest on: the fp32 matrix instructions add their k in order, each step
    one fused multiply-add, denormals kept, from +0: bit for bit at the kernels' chain lengths (one group's
    4 to 144 entries), in regimes of magnitude."""
    import ctypes

    libm = ctypes.CDLL("libm.so.6")
    libm.fmaf.argtypes, libm.fmaf.restype = [ctypes.c_float] * 3, ctypes.c_float
    rng = np.random.default_rng(rows * 10 + REGIMES.index(regime))
    print(f"[gpu-test] mfma chains rows={rows} {regime}", flush=True)
    seen = np.zeros(0, np.float32)
    for K in (4, 8, 40, 64, 144):
        for _ in range(6):
            a, b = (rng.standard_normal((rows, K)) for _ in range(2))
            if regime == "wide":
                a, b = (x * 2.0 ** rng.integers(-45, 46, x.shape) for x in (a, b))
            elif regime == "cancel":  # (each pair of terms nearly cancels)
                a[:, 1::2] = -a[:, ::2]
                b[:, 1::2] = b[:, ::2] * (1 + 2.0 ** -7 * rng.integers(-1, 2, b[:, ::2].shape))
            elif regime == "denormal_in":
                a, b = a * 2.0 ** -128, b * 2.0 ** rng.integers(-2, 100, b.shape)
            elif regime == "denormal_out":
                a, b = (x * 2.0 ** rng.integers(-75, -63, x.shape) for x in (a, b))
            elif regime == "overflow":
                a, b = (x * 2.0 ** rng.integers(58, 65, x.shape) for x in (a, b))
            elif regime == "not_finite":
                a[0, 1], b[1, 2], a[2, 3], b[2, 3] = np.inf, -np.inf, np.nan, 0.0
            a, b = a.astype(np.float32), b.astype(np.float32)
            if regime != "float32":
                a, b = (torch.from_numpy(x).bfloat16().float().numpy() for x in (a, b))
            want = fma_chain(a, b)
            x = np.float32(0)
            for k in range(K):
                x = libm.fmaf(float(a[3, k]), float(b[2, k]), float(x))
            assert bits(np.float32(x)) == bits(want[3, 2]) or np.isnan(x)
            ad, bd = torch.from_numpy(a).to(cuda), torch.from_numpy(b).to(cuda)
            out = torch.zeros(rows, rows, device=cuda)
            assert mk_build.load().lxm_t_mfma(rows, ctypes.c_void_p(ad.data_ptr()),
                                              ctypes.c_void_p(bd.data_ptr()), K,
                                              ctypes.c_void_p(out.data_ptr()), None) == 0
            got = out.cpu().numpy()
            assert ((bits(got) == bits(want)) | (np.isnan(got) & np.isnan(want))).all(), K
            seen = np.concatenate([seen, (a if regime == "denormal_in" else want).reshape(-1)])
    mag = np.abs(seen)
    if regime.startswith("denormal"):  # (the regime is what it says)
        assert ((mag > 0) & (mag < 2.0 ** -126)).mean() > 0.01
    if regime == "overflow":
        assert 0.01 < np.isinf(seen).mean() < 0.99
    if regime == "not_finite":
        assert np.isnan(seen).any() and np.isinf(seen).any()


def test_dense_prefill_full_widths(cuda):
    check_prefill(21, 3, seed=5, name="mid")


TWO_LAYERS = [9, 25, 40, 70]  # prompt lengths


@pytest.fixture(scope="module")
def wide():
    """Two layers at config 4's full widths (layer 1's states see layer 0's out_proj, SwiGLU and
    down_proj), and the oracle's states after each of the prompts below."""
    from dataclasses import replace

    from oracle import oracle as ox

    spec = replace(synth.config4_mid(), n_layers=2, vocab=256)
    dm = synth.build_dense(spec, "cpu")
    conv0, rec0 = synth.dense_state(dm, 5)
    toks = [int(x) for x in np.random.default_rng(41).integers(0, spec.vocab, 200)]
    om = ox.OracleModel(synth.to_sparse(dm))
    c, r, at, done = conv0.copy(), rec0.copy(), {}, 0
    for n in TWO_LAYERS:
        print(f"[gpu-test] the oracle's tokens {done} .. {n - 1}", flush=True)
        om.decode(c, r, toks[done:n], n - done)
        at[n], done = (c.copy(), r.copy()), n
    return synth.dense_to(dm, "cuda"), conv0, rec0, toks, at


@pytest.mark.parametrize("n", TWO_LAYERS)
def test_dense_prefill_full_widths_two_layers(cuda, wide, n):
    """Every row kernel at its real row lengths against the oracle, seen through layer 1: 16-row tiles of 16,
    32 and (hidden rows) 64 tokens, 32-row tiles with a whole and a partial token tile."""
    dm, conv0, rec0, toks, at = wide
    print(f"[gpu-test] dense prefill two full-width layers: n={n}", flush=True)
    cache = fast.StateCache(conv0, rec0, "bf16", "cuda")
    dense.DenseDecode(dm, cache).prefill(toks[:n])
    assert (bits(cache.conv_numpy()) == bits(at[n][0])).all()
    assert (bits(cache.rec_numpy()) == bits(at[n][1])).all()


@pytest.mark.parametrize("n", [64, 65, 130, 200])
def test_dense_prefill_full_widths_equals_steps(cuda, wide, n):
    """More token tiles: the states of as many forced steps."""
    dm, conv0, rec0, toks, _ = wide
    print(f"[gpu-test] dense prefill two full-width layers against steps: n={n}", flush=True)
    out = []
    for batched in (False, True):
        cache = fast.StateCache(conv0, rec0, "bf16", "cuda")
        dd = dense.DenseDecode(dm, cache, max_steps=256)
        dd.prefill(toks[:n]) if batched else dd.run(toks[:n], n)
        out.append((cache.conv_numpy(), cache.rec_numpy()))
    for a, b in zip(*out):
        assert (bits(a) == bits(b)).all()


def test_dense_prefill_equals_steps_config4(cuda):
    """At config 4's full size (24 layers, hidden 2560, vocabulary 248,320): a 40-token prompt
    through lxm_dn_prefill and one step leaves the prediction and every state and window that
    40 forced steps leave, bit for bit (two native paths, each pinned to the oracle above on the
    scaled-down stacks)."""
    spec = synth.config4()
    dm = synth.build_dense(spec, "cuda")
    d = dm.dims
    toks = [int(x) for x in np.random.default_rng(9).integers(0, spec.vocab, 40)]
    print(f"[gpu-test] dense prefill config 4 full size: T={len(toks)}", flush=True)
    out = []
    for batched in (False, True):
        conv0 = np.zeros((d.n_layers, d.n_conv, 4), np.float32)
        rec0 = np.zeros((d.n_layers, d.nv, 256, 128), np.float32)
        cache = fast.StateCache(conv0, rec0, "bf16", "cuda")
        dd = dense.DenseDecode(dm, cache, max_steps=64)
        if batched:
            dd.prefill(toks[:-1])
            p = dd.run(toks[-1:], 1)
        else:
            p = dd.run(toks, len(toks))[-1:]
        out.append((p, [l.conv_states[0].clone() for l in cache.layers],
                    [l.recurrent_states[0].clone() for l in cache.layers]))
        del dd, cache
    (p0, c0, r0), (p1, c1, r1) = out
    assert p0 == p1
    for a, b in zip(c0, c1):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))
    for a, b in zip(r0, r1):
        assert torch.equal(a.view(torch.int32), b.view(torch.int32))
    assert any(bool(r.any()) for r in r1)  # (the prompt moved the live states)


def test_dense_prefill_rejects_bad_token(cuda):
    spec, dm_cpu, _ = model()
    conv0, rec0 = synth.dense_state(dm_cpu)
    dd = dense.DenseDecode(synth.dense_to(dm_cpu, "cuda"), fast.StateCache(conv0, rec0, "bf16", "cuda"))
    with pytest.raises(ValueError, match="out of range"):
        dd.prefill([1, spec.vocab])


def test_dense_rejects_dead_state(cuda):
    """A nonzero state on a dead value head would not stay zero as the kernels assume."""
    spec, dm_cpu, sm = model()
    conv0, rec0 = synth.dense_state(dm_cpu)
    rec0[0, 2, 0, 0] = 1.0  # value head 2 of key head 0: dead (r_live = 2)
    cache = fast.StateCache(conv0, rec0, "bf16", "cuda")
    with pytest.raises(AssertionError):
        dense.DenseDecode(synth.dense_to(dm_cpu, "cuda"), cache)


def check_prefill_chunked(T, n, seed=None, name="small"):
    """lxm_dn_prefill_chunked over T - 1 tokens (the stock T > 1 path: chunks of 64, the delta
    rule on the matrix cores), then n steps from the last token, against the oracle's restatement
    of the same (ox_prefill_chunked, then ox_decode). The chunked delta rule sums in its own order
    (MFMA tiles), so its outputs match the oracle's to about 1e-6 before they round to bf16: a
    rare output rounds the other way and moves the residual by one bf16 step, which the later
    layers carry. Bounds: the first layer's recurrent states (its inputs are the embeddings, so
    only the delta rule's own arithmetic differs) within 1e-6 of each head's largest magnitude
    (measured <= 2e-7; the oracle's recurrent and chunked forms differ by up to 9e-7); later
    layers within 5e-3 (measured <= 9e-4; the oracle's two forms differ by up to 1.3e-3 there);
    at least 99 % of the conv windows' values bit for bit (measured: all) and the rest within
    2^-6 relative; the same greedy predictions."""
    from oracle import oracle as ox

    spec, dm_cpu, sm = model(name)
    conv0, rec0 = synth.dense_state(dm_cpu, seed)
    toks = [int(x) for x in np.random.default_rng(23 + T).integers(0, spec.vocab, T)]
    print(f"[gpu-test] dense chunked prefill {spec.name}: T={T} n={n} seed={seed}", flush=True)
    dm = synth.dense_to(dm_cpu, "cuda")
    cache = fast.StateCache(conv0, rec0, "bf16", "cuda")
    dd = dense.DenseDecode(dm, cache)
    dd.prefill(toks[:-1], mode="chunked")
    gc_, gr = cache.conv_numpy().copy(), cache.rec_numpy().copy()
    preds = dd.run(toks[-1:], n)
    om = ox.OracleModel(sm)
    c, r = conv0.copy(), rec0.copy()
    om.prefill_chunked(c, r, toks[:-1])
    diff = bits(gc_) != bits(c)
    assert diff.mean() <= 0.01, diff.mean()
    assert (np.abs(gc_ - c) <= 2.0 ** -6 * np.abs(c)).all()
    for L in range(r.shape[0]):
        bound = 1e-6 if L == 0 else 5e-3
        for h in range(r.shape[1]):
            ref = np.abs(r[L, h]).max()
            assert np.abs(gr[L, h] - r[L, h]).max() <= bound * max(ref, 1e-30), (L, h)
    po, _, _ = om.decode(c, r, toks[-1:], n)
    assert preds == po.tolist()
    # the prompt moved the live heads' states (the chunked path ran)
    assert not np.array_equal(gr, rec0)
    return gr


@pytest.mark.parametrize("T,seed", [(150, None), (66, 3), (20, 3)])
def test_dense_prefill_chunked_small(cuda, T, seed):
    """Chunks of 64 with a ragged last one, exactly one chunk plus a token, a prompt shorter than
    one chunk; from zero and from live states."""
    check_prefill_chunked(T, 6, seed=seed)


def test_dense_prefill_chunked_full_widths(cuda):
    check_prefill_chunked(70, 3, seed=5, name="mid")


def test_dense_prefill_chunked_close_to_batched(cuda):
    """The chunked and the batched (recurrent, bit-exact to forced steps) prompts on the same
    tokens: the same states up to rounding: the first layer within 2e-6 of each head's largest
    magnitude (the two forms' own arithmetic), the later ones within 5e-3 (rare bf16 outputs
    rounding the other way, carried)."""
    spec, dm_cpu, sm = model("small")
    conv0, rec0 = synth.dense_state(dm_cpu, 3)
    toks = [int(x) for x in np.random.default_rng(5).integers(0, spec.vocab, 100)]
    dm = synth.dense_to(dm_cpu, "cuda")
    out = []
    for mode in ("batched", "chunked"):
        cache = fast.StateCache(conv0, rec0, "bf16", "cuda")
        dense.DenseDecode(dm, cache).prefill(toks, mode=mode)
        out.append(cache.rec_numpy())
    a, b = out
    for L in range(a.shape[0]):
        bound = 2e-6 if L == 0 else 5e-3
        for h in range(a.shape[1]):
            assert np.abs(a[L, h] - b[L, h]).max() <= bound * max(np.abs(a[L, h]).max(), 1e-30)
    assert not np.array_equal(a, b)  # different forms, different roundings
