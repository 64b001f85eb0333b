"""The stock forward's chunked delta rule on the matrix cores (csrc/lxm_chunk.hip, C ABI
include/lxm_chunk.h): torch_chunk_gated_delta_rule (transformers qwen3_5 :249-327; the reference's
fla chunk_gated_delta_rule call, lx/lx/fast.py:342-345) for value heads over T positions, in
chunks of 64 from position 0, the state carried from chunk to chunk.

    o = gated_delta_chunked(q, k, v, g, beta, S)   # S updated in place
"""

from __future__ import annotations

import ctypes

import torch

from . import mk_build

CHUNK = 64
CHUNK_WS = 76304       # bytes of workspace per (value head, chunk) (LXM_CHUNK_WS)
WS_MAX = 160 << 20     # a call's workspace at most (68 chunks of 32 heads; more go in groups)


def workspace(n_slots: int, T: int, device) -> torch.Tensor:
    """The workspace of a T-position call (lxm_gdn_chunks): every chunk's, or what WS_MAX holds."""
    nch = (T + CHUNK - 1) // CHUNK
    per = n_slots * CHUNK_WS
    return torch.empty(per * max(1, min(nch, WS_MAX // max(1, per))), dtype=torch.uint8, device=device)


class ChunkIO(ctypes.Structure):
    _fields_ = [(n, ctypes.c_void_p) for n in ("q", "k", "v", "beta", "g", "S", "o")] + \
        [(n, ctypes.c_int64) for n in ("qk_ts", "qk_hs", "v_ts", "g_ts", "g_hs", "gl_ts", "o_ts")] + \
        [(n, ctypes.c_int32) for n in ("n", "n_slots", "rl", "rfull", "kl", "o_bf16")]


@torch.no_grad()
def gated_delta_chunked(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, g: torch.Tensor,
                        beta: torch.Tensor, S: torch.Tensor, kl: int = 128,
                        o_bf16: bool = False) -> torch.Tensor:
    """q, k (T, nk, 256) float32 (l2-normed; q already times 1/16), v (T, nv, 128), g (T, nv) log
    decays, beta (T, nv), S (nv, 256, 128) float32 updated in place (value head h reads key head
    h // (nv // nk)). Only the first kl key dims may be nonzero. Returns o (T, nv, 128) float32."""
    lib = mk_build.load()
    T, nk, K = q.shape
    nv = v.shape[1]
    assert K == 256 and v.shape == (T, nv, 128) and k.shape == q.shape
    assert g.shape == (T, nv) and beta.shape == (T, nv) and S.shape == (nv, 256, 128)
    assert nv % nk == 0 and 0 < kl <= 128 and kl % 16 == 0
    for t in (q, k, v, g, beta, S):
        assert t.dtype == torch.float32 and t.is_contiguous() and t.is_cuda
    o = torch.empty(T, nv, 128, dtype=torch.float32, device=q.device)
    if T == 0:
        return o
    st = ctypes.c_void_p(torch.cuda.current_stream(q.device).cuda_stream)
    io = ChunkIO(q=q.data_ptr(), k=k.data_ptr(), v=v.data_ptr(), beta=beta.data_ptr(),
                 g=g.data_ptr(), S=S.data_ptr(), o=o.data_ptr(), qk_ts=nk * 256, qk_hs=256,
                 v_ts=nv * 128, g_ts=nv, g_hs=1, gl_ts=nv, o_ts=nv * 128, n=min(T, CHUNK),
                 n_slots=nv, rl=nv // nk, rfull=nv // nk, kl=kl, o_bf16=int(o_bf16))
    if T <= CHUNK:  # (one launch, no workspace)
        e = lib.lxm_gdn_chunk(ctypes.byref(io), st)
    else:
        ws = workspace(nv, T, q.device)
        e = lib.lxm_gdn_chunks(ctypes.byref(io), T, ctypes.c_void_p(ws.data_ptr()), ws.numel(), st)
    if e:
        raise RuntimeError(f"lxm_gdn_chunk failed: hipError {e}")
    return o
