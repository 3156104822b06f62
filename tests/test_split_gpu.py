"""Calls whose key segments are split into chunks over workgroups of their own (few query rows against
long ``cu_seqlens_k`` segments): parity with the oracle at every chunk edge, the unsplit kernels' bits
where a row reads one chunk, and graph replay."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from conftest import announce

pytestmark = pytest.mark.gpu

# keys around the 256-key chunk and the 64- and 32-key tiles; tails of one row, a part of a tile, a
# tile and a row, none, and a tail longer than its keys (its first rows reach no key)
KEYS = [1537, 256, 255, 257, 1024, 2100, 64, 0, 1600, 300, 2]
TAILS = [1, 5, 32, 33, 16, 17, 64, 3, 0, 70, 9]
# (head_dim, query heads, kv heads, window, causal, gate)
CASES = [
    (64, 4, 4, (-1, -1), True, False),
    (64, 8, 2, (-1, 3), False, True),
    (64, 6, 3, (1700, -1), True, False),
    (128, 8, 2, (-1, -1), True, True),
    (128, 4, 2, (-1, -1), False, False),
    (128, 5, 5, (900, 900), False, False),
    (256, 8, 2, (-1, -1), True, True),
    (256, 4, 2, (-1, -1), False, False),
    (256, 3, 3, (1600, -1), True, False),
]


def _inputs(d, hq, hkv, gate, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)

    def draw(t, h):
        return torch.randn(t, h, d, generator=g, device="cuda").bfloat16()

    q, k, v = draw(sum(TAILS), hq), draw(sum(KEYS), hkv), draw(sum(KEYS), hkv)
    return q, k, v, draw(sum(TAILS), hq) if gate else None


def _cu(lengths):
    return torch.tensor([0, *np.cumsum(lengths).tolist()], dtype=torch.int32, device="cuda")


def _call(pe, case, q, k, v, gate, out, bytes_, short_max=-1):
    """The call through the C entry point with a workspace of `bytes_(chunks, size)` bytes."""
    from packed_encoders_amd import _lib
    from packed_encoders_amd.hip_attention import _args

    d, _, _, window, causal, _ = case
    lib, cu, cuk = _lib.library(), _cu(TAILS), _cu(KEYS)
    a = _args(q, k, v, out, cu, max(TAILS), d ** -0.5, *window, causal, gate, short_max, cu_k=cuk, max_seqlen_k=max(KEYS))
    size = ctypes.c_size_t()
    assert lib.pe_attn_workspace_size(ctypes.byref(a), ctypes.byref(size)) == 0
    n = bytes_(lib.pe_attn_key_chunks(ctypes.byref(a)), size.value)
    ws = torch.full((n,), 0xFF, dtype=torch.uint8, device="cuda")  # partial rows nobody wrote would be NaN
    assert lib.pe_varlen_attn_fwd(ctypes.byref(a), ws.data_ptr(), n, torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("case", CASES, ids=str)
def test_split_call_matches_the_oracle_and_the_unsplit_kernel(pe, case):
    announce(f"split {case}")
    d, hq, hkv, window, causal, gated = case
    q, k, v, gate = _inputs(d, hq, hkv, gated, seed=d + hq)
    chunks = []
    split = _call(pe, case, q, k, v, gate, torch.full_like(q, 7.0), lambda c, n: chunks.append(c) or n)
    assert chunks == [9]  # 2,100 keys in chunks of 256, the smallest
    # a workspace for the list alone (at most one entry per 16-row tile of each segment); a split call
    # routes nothing to the short kernel by default
    plain = _call(pe, case, q, k, v, gate, torch.full_like(q, 7.0), lambda c, n: 256 + 16 * len(KEYS) * 5, 0)
    routed = _call(pe, case, q, k, v, gate, torch.full_like(q, 7.0), lambda c, n: n, 32 if d <= 128 else 0)
    want = pe.runtime_attention.oracle_attention(q, k, v, TAILS, KEYS, causal, window)
    if gate is not None:
        want = want * torch.sigmoid(gate.double())
    for got in (split, plain, routed):
        assert (got.double() - want).abs().max() <= 2e-2
        cos = torch.nn.functional.cosine_similarity(got.double().flatten(1), want.flatten(1), dim=-1)
        seen = want.abs().amax(dim=(1, 2)) > 0
        assert cos[seen].min() >= 0.9999
    at = 0
    for tail, keys in zip(TAILS, KEYS):
        if keys <= 256:
            assert torch.equal(split[at:at + tail], plain[at:at + tail]), (tail, keys)
        at += tail


def test_small_reaches_and_full_chips_stay_unsplit(pe):
    """The rule, from host sizes alone: a window that spans few keys, a call whose tiles fill the
    chip, shared key segments, strips and unbounded head_dim 64 calls are not split."""
    from packed_encoders_amd import _lib

    lib = _lib.library()

    def chunks(d=128, n=8, tail=16, keys=4096, hq=32, hkv=8, own=True, **kw):
        a = _lib.AttnArgs()
        a.struct_size, a.dtype = ctypes.sizeof(_lib.AttnArgs), 1
        a.n_seq, a.total_tokens, a.max_seqlen = n, n * tail, tail
        a.n_heads_q, a.n_heads_kv, a.head_dim, a.softmax_scale = hq, hkv, d, d ** -0.5
        a.window_left, a.window_right, a.causal, a.short_max = -1, -1, 1, -1
        if own:
            a.cu_seqlens_k, a.total_tokens_k, a.max_seqlen_k = 8, n * keys, keys
        for name, value in kw.items():
            setattr(a, name, value)
        return lib.pe_attn_key_chunks(ctypes.byref(a))

    assert chunks() == 7 and chunks(n=1) == 16 and chunks(keys=1537, n=1) == 7 and chunks(n=64, tail=1) == 3
    assert chunks(d=256, n=4) == 13
    assert chunks(keys=1536) == chunks(own=False) == chunks(n=65) == chunks(tail=65, n=32) == 1
    # a full chip of equal walks: split only where the partial rows cost nothing (64 x 4,096 keys, unsplit
    # and split: 16-row tails 208 and 243 us, one row 215 and 202; 64 x 2,304 129 and 146, 125 and 120)
    assert chunks(n=64) == chunks(keys=2304, n=64) == chunks(keys=2200, n=64) == 1
    assert chunks(n=64, tail=1) == 3 and chunks(keys=2304, n=64, tail=1) == 2
    assert chunks(window_left=1000) == 1 and chunks(window_left=1600) == 7
    assert chunks(strip=2) == 1 and chunks(d=64, causal=0) == 1 and chunks(d=64, n=1) == 16
    assert chunks(head_dim=96) == -2


def test_split_call_of_many_segments_is_planned(pe):
    """More segments than a wave numbers: the split kernel reads the plan's list."""
    announce("split call of 300 segments")
    rng = np.random.default_rng(3)
    keys, tails = rng.integers(0, 40, size=300), rng.integers(0, 3, size=300)
    keys[[0, 150, 299]], tails[[0, 150, 299]] = [1700, 2100, 1537], [2, 1, 2]
    g = torch.Generator(device="cuda").manual_seed(3)
    q, k, v = (torch.randn(int(t), h, 128, generator=g, device="cuda").bfloat16()
               for t, h in ((tails.sum(), 4), (keys.sum(), 1), (keys.sum(), 1)))
    with torch.inference_mode():
        got = pe.varlen_attention(q, k, v, _cu(tails), 2, causal=True, cu_seqlens_k=_cu(keys), max_seqlen_k=2100)
    want = pe.runtime_attention.oracle_attention(q, k, v, tails, keys, True)
    assert (got.double() - want).abs().max() <= 2e-2
    from packed_encoders_amd import _lib
    from packed_encoders_amd.hip_attention import _args

    a = _args(q, k, v, got, _cu(tails), 2, 128 ** -0.5, -1, -1, True, None, -1, cu_k=_cu(keys), max_seqlen_k=2100)
    assert _lib.library().pe_attn_key_chunks(ctypes.byref(a)) > 1  # it did split


def _edge_batch(d, hq, hkv, n, chunk):
    """Tails and key lengths of n segments whose call is cut into chunks of `chunk` keys: segments at the
    chunk's edges, none, few and many keys, and the others sized so that the rule gives that chunk."""
    g = np.gcd(hq // hkv, 4)
    bm = (64 if d == 256 else 128) // g
    groups, slots = n * hq // g, (3 if d == 64 else 2) * 256
    mean = (chunk - 32) * (slots * 7 // 4 - groups) // (2 * groups)
    edges = [chunk - 1, chunk, chunk + 1, 2 * chunk - 1, 2 * chunk, 2 * chunk + 1, 0, 1, 63, 65, max(1700, 3 * chunk)]
    rng = np.random.default_rng(d + n + chunk)
    rest = (mean - 1) * n - sum(edges)
    assert rest > 0
    others = rng.multinomial(rest, rng.dirichlet(np.full(n - len(edges), 8.0)))
    order = rng.permutation(n)
    keys = np.array(edges + others.tolist())[order]
    tails = np.array([(bm, 1, bm - 1, 2, 5)[i % 5] for i in range(n - 1)] + [0])[order]
    return keys.tolist(), tails.tolist()


# head_dim, query heads, kv heads, segments (360 workgroups of the unsplit call), window, causal, gate
EDGE_CASES = [
    (64, 8, 8, 45, (-1, -1), True, True), (64, 8, 4, 90, (2500, 1500), False, False), (64, 8, 2, 180, (3400, -1), True, True),
    (128, 8, 8, 45, (-1, -1), False, False), (128, 8, 4, 90, (-1, -1), True, True), (128, 8, 2, 180, (900, 900), False, True),
    (256, 8, 8, 45, (3000, -1), True, False), (256, 8, 4, 90, (-1, -1), False, True), (256, 8, 2, 180, (-1, -1), True, False),
]


@pytest.mark.parametrize("chunk", [320, 640, 1152])
@pytest.mark.parametrize("case", EDGE_CASES, ids=str)
def test_split_instances_at_their_chunk_edges(pe, case, chunk):
    """Every head_dim and heads per workgroup, gated and not, with chunks under 1,024 keys (the kernels
    find their tiles) and past it (they read the plan, which the workspace's header tells)."""
    from packed_encoders_amd import _lib
    from packed_encoders_amd.hip_attention import _args

    d, hq, hkv, n, window, causal, gated = case
    announce(f"split chunk {chunk} {case}")
    keys, tails = _edge_batch(d, hq, hkv, n, chunk)
    g = torch.Generator(device="cuda").manual_seed(d + chunk)
    q, k, v, gt = (torch.randn(t, h, d, generator=g, device="cuda").bfloat16()
                   for t, h in ((sum(tails), hq), (sum(keys), hkv), (sum(keys), hkv), (sum(tails), hq)))
    lib, cu, cuk, stream = _lib.library(), _cu(tails), _cu(keys), torch.cuda.current_stream().cuda_stream
    outs, header = [], None
    for size_of in (lib.pe_attn_workspace_size, lib.pe_attn_plan_size):  # split, unsplit
        out = torch.full_like(q, 7.0)
        a = _args(q, k, v, out, cu, max(tails), d ** -0.5, *window, causal, gt if gated else None, 0, cu_k=cuk,
                  max_seqlen_k=max(keys))
        assert lib.pe_attn_key_chunks(ctypes.byref(a)) == -(-max(keys) // chunk) > 1
        size = ctypes.c_size_t()
        assert size_of(ctypes.byref(a), ctypes.byref(size)) == 0
        ws = torch.full((size.value,), 0xFF, dtype=torch.uint8, device="cuda")  # unwritten partial rows are NaN
        assert lib.pe_varlen_attn_fwd(ctypes.byref(a), ws.data_ptr(), size.value, stream) == 0
        torch.cuda.synchronize()
        outs.append(out)
        header = ws[:8].view(torch.int32).tolist() if header is None else header
    assert header == [-1, -1] if chunk < 1024 else header[0] == header[1] == sum(t > 0 for t in tails)
    want = pe.runtime_attention.oracle_attention(q, k, v, tails, keys, causal, window)
    if gated:
        want = want * torch.sigmoid(gt.double())
    at = 0
    for tail, length in zip(tails, keys):
        part = slice(at, at + tail)
        if length <= chunk:
            assert torch.equal(outs[0][part], outs[1][part]), (tail, length)
        at += tail
    for got in outs:
        assert (got.double() - want).abs().max() <= 2e-2


@pytest.mark.parametrize("d", [64, 128, 256])
def test_split_call_replays_in_a_graph(pe, d):
    announce(f"split call in a graph, head_dim {d}")
    q, k, v, _ = _inputs(d, 8, 2, False, seed=d)
    cu, cuk = _cu(TAILS), _cu(KEYS)

    def call():
        return pe.varlen_attention(q, k, v, cu, max(TAILS), causal=True, cu_seqlens_k=cuk, max_seqlen_k=max(KEYS))

    with torch.inference_mode():
        want = [call()]
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = call()
        for i in range(4):
            if i % 2:
                k.neg_()
                want.append(call())
                torch.cuda.synchronize()
            out.fill_(7.0)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want[-1]), i


def test_split_calls_on_two_streams_share_nothing(pe):
    """Calls in one shared_plans scope on two streams at once give the bits of the calls alone."""
    announce("split calls on two streams")
    a, b = _inputs(128, 8, 2, False, seed=1), _inputs(128, 8, 2, False, seed=2)
    cu, cuk = _cu(TAILS), _cu(KEYS)

    def call(t):
        return pe.varlen_attention(t[0], t[1], t[2], cu, max(TAILS), causal=True, cu_seqlens_k=cuk,
                                   max_seqlen_k=max(KEYS))

    with torch.inference_mode():
        want = call(a), call(b)
        streams = torch.cuda.Stream(), torch.cuda.Stream()
        torch.cuda.synchronize()
        with pe.shared_plans():
            got = ([], [])
            for _ in range(6):
                for stream, t, outs in zip(streams, (a, b), got):
                    with torch.cuda.stream(stream):
                        outs.append(call(t))
            torch.cuda.synchronize()
    for w, outs in zip(want, got):
        assert all(torch.equal(w, o) for o in outs)


def _chunks(n, tail, keys, bound, hq=32, hkv=8, d=128):
    from packed_encoders_amd import _lib

    a = _lib.AttnArgs()
    a.struct_size, a.dtype = ctypes.sizeof(_lib.AttnArgs), 1
    a.n_seq, a.total_tokens, a.max_seqlen = n, n * tail, tail
    a.n_heads_q, a.n_heads_kv, a.head_dim, a.softmax_scale = hq, hkv, d, d ** -0.5
    a.window_left, a.window_right, a.causal, a.short_max = -1, -1, 1, -1
    a.cu_seqlens_k, a.total_tokens_k, a.max_seqlen_k = 8, n * keys, bound
    return _lib.library().pe_attn_key_chunks(ctypes.byref(a))


def test_a_bound_far_above_the_lengths_adds_no_chunks(pe):
    """max_seqlen_k may be a capacity: no segment holds more keys than the call, and the workgroups of
    chunks that a segment does not have stay few."""
    assert _chunks(1, 1, 500, 131072) == 1  # 500 keys in all: nothing to split
    assert _chunks(16, 1, 1000, 131072) == _chunks(16, 1, 1000, 16000) <= 42
    assert _chunks(32, 1, 300, 8192) * 32 * 8 <= 8 * 512 + 32 * 8  # eight rounds of two workgroups per CU
    assert _chunks(1, 1, 8192, 131072) == _chunks(1, 1, 8192, 8192) == 32


@pytest.mark.parametrize("d", [64, 128, 256])
def test_split_call_under_a_loose_bound(pe, d):
    announce(f"split call, max_seqlen_k a capacity, head_dim {d}")
    q, k, v, _ = _inputs(d, 8, 2, False, seed=d)
    with torch.inference_mode():
        got = pe.varlen_attention(q, k, v, _cu(TAILS), max(TAILS), causal=True, cu_seqlens_k=_cu(KEYS),
                                  max_seqlen_k=1 << 20)
    want = pe.runtime_attention.oracle_attention(q, k, v, TAILS, KEYS, True)
    assert (got.double() - want).abs().max() <= 2e-2


@pytest.mark.parametrize("case", [CASES[0], CASES[3], CASES[6]], ids=str)
def test_staged_call_needs_the_plan_alone(pe, case):
    """The staged entry points over a workspace of pe_attn_plan_size, and the whole call with it: unsplit,
    bit for bit alike."""
    from packed_encoders_amd import _lib
    from packed_encoders_amd.hip_attention import _args

    announce(f"staged call over the plan alone {case}")
    d, hq, hkv, window, causal, gated = case
    q, k, v, gate = _inputs(d, hq, hkv, gated, seed=d)
    lib, cu, cuk, out = _lib.library(), _cu(TAILS), _cu(KEYS), torch.full_like(q, 7.0)
    a = _args(q, k, v, out, cu, max(TAILS), d ** -0.5, *window, causal, gate, 0, cu_k=cuk, max_seqlen_k=max(KEYS))
    size, ref, stream = ctypes.c_size_t(), ctypes.byref(a), torch.cuda.current_stream().cuda_stream
    assert lib.pe_attn_plan_size(ref, ctypes.byref(size)) == 0 and lib.pe_attn_key_chunks(ref) > 1
    guard = torch.full((size.value + 4096,), 0xAA, dtype=torch.uint8, device="cuda")
    assert lib.pe_attn_plan(ref, guard.data_ptr(), size.value, stream) == 0
    assert lib.pe_attn_short_fwd(ref, stream) == 0
    assert lib.pe_attn_tiled_fwd(ref, guard.data_ptr(), size.value, stream) == 0
    torch.cuda.synchronize()
    assert (guard[size.value:] == 0xAA).all()
    whole = _call(pe, case, q, k, v, gate, torch.full_like(q, 7.0), lambda chunks, n: size.value, 0)
    assert torch.equal(out, whole)

@pytest.mark.parametrize("hq,hkv", [(8, 1), (12, 4), (12, 2), (5, 1), (8, 2)])
@pytest.mark.parametrize("d", [64, 128, 256])
def test_split_calls_whose_workgroups_share_keys(pe, d, hq, hkv):
    """Head groups of one kv head (two, three, three, five, one) and tails of up to three query tiles, ragged and
    empty ones among them: workgroups that share keys are dealt to one XCD, every row is written once."""
    from packed_encoders_amd import _lib
    from packed_encoders_amd.hip_attention import _args

    bm = (64 if d == 256 else 128) // int(np.gcd(hq // hkv, 4))
    lib, stream = _lib.library(), torch.cuda.current_stream().cuda_stream
    for tails in ([1] * 11, [3 * bm, 2 * bm + 1, bm, 0, 3 * bm - 1, 1, 2 * bm, 2 * bm - 1, 3 * bm], [2 * bm] * 8):
        announce(f"split, shared keys, head_dim {d}, heads {hq}:{hkv}, tails {tails}")
        keys = [3000 - 211 * i for i in range(len(tails))]
        g = torch.Generator(device="cuda").manual_seed(d + hq)
        q, k, v = (torch.randn(t, h, d, generator=g, device="cuda").bfloat16()
                   for t, h in ((sum(tails), hq), (sum(keys), hkv), (sum(keys), hkv)))
        cu, cuk, out, size = _cu(tails), _cu(keys), torch.full_like(q, 7.0), ctypes.c_size_t()
        a = _args(q, k, v, out, cu, max(tails), d ** -0.5, -1, -1, True, None, 0, cu_k=cuk, max_seqlen_k=max(keys))
        assert lib.pe_attn_workspace_size(ctypes.byref(a), ctypes.byref(size)) == 0
        assert lib.pe_attn_key_chunks(ctypes.byref(a)) > 1
        ws = torch.full((size.value,), 0xFF, dtype=torch.uint8, device="cuda")  # unwritten partial rows are NaN
        assert lib.pe_varlen_attn_fwd(ctypes.byref(a), ws.data_ptr(), size.value, stream) == 0
        torch.cuda.synchronize()
        want = pe.runtime_attention.oracle_attention(q, k, v, tails, keys, True)
        assert (out.double() - want).abs().max() <= 2e-2
