"""The chunked delta rule on the matrix cores (lxm_gdn_chunk) against the oracle's restatement of
torch_chunk_gated_delta_rule, on an MI355X, through the C ABI.

Random regime: outputs and final states within 2e-6 of each head's largest magnitude (the MFMA
tiles and the blocked triangular inverse sum in their own orders; the oracle itself is within 1e-6
of transformers' function, tests/test_oracle.py). Exact regime (one-hot keys and queries, beta in
{0, 1}, no decay, dyadic values): bit for bit. Sequences of one partial chunk, whole chunks and a
ragged tail; several key heads with several value heads each.
"""

import numpy as np
import pytest
import torch

from linuxformer_amd import mk_build
from linuxformer_amd.chunk import gated_delta_chunked

pytestmark = pytest.mark.gpu

TOL = 2e-6


@pytest.fixture(scope="module")
def cuda():
    assert torch.cuda.is_available(), "the gpu tests need an MI355X"
    mk_build.load()
    return torch.device("cuda", 0)


def _inputs(T, nk, R, seed, exact=False):
    from golden.make_golden import chunk_inputs

    nv = nk * R
    q = np.zeros((T, nk, 256), np.float32)
    k = np.zeros((T, nk, 256), np.float32)
    v = np.zeros((T, nv, 128), np.float32)
    g = np.zeros((T, nv), np.float32)
    beta = np.zeros((T, nv), np.float32)
    S = np.zeros((nv, 256, 128), np.float32)
    for kh in range(nk):
        qi, ki, _, _, _, _ = chunk_inputs(T, seed + 100 * kh, exact)
        q[:, kh], k[:, kh] = qi, ki
    for vh in range(nv):
        _, _, vi, gi, bi, Si = chunk_inputs(T, seed + 7 * vh + 1, exact)
        v[:, vh], g[:, vh], beta[:, vh], S[vh] = vi, gi, bi, Si
    return q, k, v, g, beta, S


def _oracle(q, k, v, g, beta, S, R):
    from oracle import oracle as ox

    T, nv = v.shape[0], v.shape[1]
    o = np.zeros((T, nv, 128), np.float32)
    S = S.copy()
    for vh in range(nv):
        Sv = np.ascontiguousarray(S[vh])
        o[:, vh] = ox.chunk_gdr(q[:, vh // R], k[:, vh // R], v[:, vh], g[:, vh], beta[:, vh], Sv, 64)
        S[vh] = Sv
    return o, S


def _run(cuda, q, k, v, g, beta, S):
    t = [torch.from_numpy(np.ascontiguousarray(a)).to(cuda) for a in (q, k, v, g, beta, S)]
    t[0] = t[0] * 0.0625  # the kernel takes the query already scaled by 1/sqrt(256)
    o = gated_delta_chunked(*t)
    torch.cuda.synchronize()
    return o.cpu().numpy(), t[5].cpu().numpy()


@pytest.mark.parametrize("T,nk,R", [(37, 1, 1), (64, 2, 2), (200, 4, 2), (130, 16, 2)])
def test_chunk_random_regime(cuda, T, nk, R):
    print(f"[gpu-test] chunk random T={T} nk={nk} R={R}", flush=True)
    q, k, v, g, beta, S = _inputs(T, nk, R, 3)
    o_ref, S_ref = _oracle(q, k, v, g, beta, S, R)
    o, Sg = _run(cuda, q, k, v, g, beta, S)
    for vh in range(nk * R):
        assert np.abs(o[:, vh] - o_ref[:, vh]).max() <= TOL * np.abs(o_ref[:, vh]).max()
        assert np.abs(Sg[vh] - S_ref[vh]).max() <= TOL * np.abs(S_ref[vh]).max()
    assert not Sg[:, 128:].any()


@pytest.mark.parametrize("T", [50, 192])
def test_chunk_exact_regime_bit_exact(cuda, T):
    print(f"[gpu-test] chunk exact T={T}", flush=True)
    q, k, v, g, beta, S = _inputs(T, 2, 2, 9, exact=True)
    o_ref, S_ref = _oracle(q, k, v, g, beta, S, 2)
    o, Sg = _run(cuda, q, k, v, g, beta, S)
    assert (o == o_ref).all()
    assert (Sg == S_ref).all()
    assert np.abs(o_ref).max() > 0


@pytest.mark.parametrize("T,nk,R,kl,groups", [(65, 1, 1, 128, 1), (200, 3, 2, 112, 2),
                                              (320, 2, 1, 16, 5), (129, 9, 1, 64, 1)])
def test_chunks_equal_single_chunks(cuda, T, nk, R, kl, groups):
    """A sequence's chunks at once (lxm_gdn_chunks: what needs no state in parallel, then the chunks in
    order; in groups of chunks when the workspace is smaller) leave the bits of one lxm_gdn_chunk call
    per chunk: ragged last chunks of one and eight positions, few key dims, odd head counts."""
    import ctypes

    from linuxformer_amd import chunk

    print(f"[gpu-test] chunks T={T} nk={nk} R={R} kl={kl} groups={groups}", flush=True)
    q, k, v, g, beta, S = (torch.from_numpy(a).to(cuda) for a in _inputs(T, nk, R, 11))
    q[..., kl:] = 0
    k[..., kl:] = 0
    S[:, kl:] = 0
    S1, S2, nv = S.clone(), S.clone(), nk * R
    parts = [gated_delta_chunked(*(t[i:i + 64].contiguous() for t in (q, k, v, g, beta)), S1, kl=kl)
             for i in range(0, T, 64)]
    o = torch.empty(T, nv, 128, device=cuda)
    io = chunk.ChunkIO(q=q.data_ptr(), k=k.data_ptr(), v=v.data_ptr(), beta=beta.data_ptr(),
                       g=g.data_ptr(), S=S2.data_ptr(), o=o.data_ptr(), qk_ts=nk * 256, qk_hs=256,
                       v_ts=nv * 128, g_ts=nv, g_hs=1, gl_ts=nv, o_ts=nv * 128, n=64, n_slots=nv,
                       rl=R, rfull=R, kl=kl, o_bf16=0)
    ws = chunk.workspace(nv, 64 * (-(-T // 64) // groups), cuda)
    lib = mk_build.load()
    e = lib.lxm_gdn_chunks(ctypes.byref(io), T, ctypes.c_void_p(ws.data_ptr()), ws.numel(), None)
    assert e == 0
    torch.cuda.synchronize()
    assert torch.equal(torch.cat(parts), o) and torch.equal(S1, S2)
    assert lib.lxm_gdn_chunks(ctypes.byref(io), T, ctypes.c_void_p(ws.data_ptr()),
                              chunk.CHUNK_WS * nv - 1, None) != 0  # (a workspace too small)


@pytest.mark.parametrize("T", [10, 65])
def test_chunk_refuses_no_heads(cuda, T):
    z = [torch.zeros(T, *n, device=cuda) for n in ((2, 256), (2, 256), (0, 128), (0,), (0,))]
    with pytest.raises(RuntimeError, match="hipError"):
        gated_delta_chunked(*z, torch.zeros(0, 256, 128, device=cuda))


@pytest.mark.parametrize("T,nk,R,kl", [(64, 33, 1, 128), (1, 20, 2, 128), (61, 32, 2, 112), (17, 13, 5, 16)])
def test_chunk_many_heads_equal_few(cuda, T, nk, R, kl):
    """One chunk of more than 32 value heads (32 state columns a workgroup) leaves the bits of calls of
    one key head each (16 columns): whole and ragged chunks, head counts off the XCDs' 8."""
    print(f"[gpu-test] chunk heads T={T} nk={nk} R={R} kl={kl}", flush=True)
    q, k, v, g, beta, S = (torch.from_numpy(a).to(cuda) for a in _inputs(T, nk, R, 5))
    q[..., kl:] = 0
    k[..., kl:] = 0
    S[:, kl:] = 0
    S1 = S.clone()
    o = gated_delta_chunked(q, k, v, g, beta, S1, kl=kl)
    for h in range(nk):
        hv = slice(h * R, h * R + R)
        S2 = S[hv].clone()
        o2 = gated_delta_chunked(*(t[:, h:h + 1].contiguous() for t in (q, k)),
                                 *(t[:, hv].contiguous() for t in (v, g, beta)), S2, kl=kl)
        assert torch.equal(o[:, hv], o2) and torch.equal(S1[hv], S2), h


def test_chunk_time_past_one_workgroup_a_cu(cuda):
    """64 heads' chunk takes no second round of workgroups (32 heads' 16-column ones are one a CU already):
    1.2 times 32 heads' time, where two rounds are 1.9 times."""
    us = {}
    for nk in (16, 32):
        args = [torch.from_numpy(a).to(cuda) for a in _inputs(64, nk, 2, 3)]
        best = []
        for _ in range(20):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(50):
                gated_delta_chunked(*args)
            b.record()
            torch.cuda.synchronize()
            best.append(a.elapsed_time(b) * 20)
        us[nk] = min(best)
    print(f"[gpu-test] chunk of 32 heads {us[16]:.1f} us, of 64 {us[32]:.1f}", flush=True)
    assert us[32] < 1.5 * us[16], us
