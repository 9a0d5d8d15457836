"""GPU parity of the prefill kernel (csrc/pkv_prefill.hip: many query rows per KV head) against the
fp64 oracle, at the edges of its row blocks (128 rows, 32 per wave), tiles (64 tokens, blocks of
32) and shares: rows and lengths on both sides of each, empty and very short rows, streams cut
into many parts and streams that fit one share, every head_dim and cache type, each mask, and
NaN bytes everywhere no query sees.

The library takes the kernel for calls with enough work, judged from the block table's width; the
cases here widen the table instead of the rows, and check that the call's plan is the prefill
kernel's (its workspace is 2 partial slots of 128 rows per workgroup).  Tolerances are the
decode's (test_gpu_fp8.assert_close): the kernel carries the same precision.
"""
from __future__ import annotations

import math

import numpy as np
import pytest

import pkv_oracle as po
from conftest import gpu_available, make_case, rand_bits
from test_gpu_fp8 import REL, assert_close, f32, fp8_cache, from_dev8, i32, to_dev8
from test_gpu_lse import assert_lse, lse_buffer
from test_gpu_parity import TOL, announce, from_dev, to_dev, torch_mod

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]

# H, Hk, D, P, lens, M, options
CASES = [
    (8, 2, 128, 16, [700, 130, 129, 1], 33, dict(causal=True)),
    (28, 4, 128, 64, [64, 65, 1000], 37, dict(causal=True, dtype=0)),          # group 7: rows end inside a block
    (4, 4, 128, 8, [257, 300], 129, dict(causal=True)),                        # one query row past a block
    (16, 1, 128, 256, [2100], 16, dict(causal=False)),                         # one stream pair, many parts
    (8, 2, 128, 32, [40, 20, 0], 64, dict(causal=True)),                       # more queries than keys
    (8, 2, 128, 16, [900, 500], 64, dict(causal=True, window=(300, 0), alibi=True)),
    (8, 2, 128, 16, [900, 31], 40, dict(causal=False, window=(400, 5), softcap=20.0)),
    (8, 2, 128, 16, [600, 333], 40, dict(causal=True, leftpad=[95, 333])),
    (8, 2, 128, 64, [600, 95], 40, dict(causal=True, fp8=True)),
    (8, 2, 128, 64, [600, 95], 40, dict(causal=True, fp8=True, dtype=0, leftpad=[33, 0], scale=-0.1)),
    (8, 8, 64, 16, [95, 96, 97, 640], 70, dict(causal=True)),
    (8, 2, 64, 8, [700, 31], 40, dict(causal=True, fp8=True, alibi=True)),
    (8, 2, 256, 16, [700, 33, 1], 40, dict(causal=True, dtype=0)),
    (4, 2, 256, 32, [400, 320], 100, dict(causal=True, window=(390, 0), softcap=30.0)),
    (8, 2, 256, 64, [300, 65], 40, dict(causal=True, fp8=True)),
    # Every layout of the capped slots, past the masked blocks of a row's end; with ALiBi every block is
    # capped ahead of them.
    (8, 2, 64, 16, [700, 130], 40, dict(causal=True, softcap=8.0)),
    (8, 2, 64, 16, [700, 130], 40, dict(causal=True, softcap=8.0, dtype=0)),
    (8, 2, 64, 16, [700, 130], 40, dict(causal=True, softcap=8.0, fp8=True)),
    (8, 2, 128, 16, [700, 130], 40, dict(causal=True, softcap=8.0, fp8=True, dtype=0)),
    (8, 2, 256, 16, [700, 130], 40, dict(causal=True, softcap=8.0, fp8=True)),
    (8, 2, 64, 16, [700, 130], 40, dict(causal=False, softcap=8.0, alibi=True)),
    (8, 2, 64, 16, [700, 130], 40, dict(causal=True, dtype=0)),
    # One query token, many heads per KV head: a decode step of the same kernel.
    (128, 1, 128, 16, [900, 1, 0, 333], 1, dict(causal=False)),
    (142, 2, 64, 64, [900, 65], 1, dict(causal=True, dtype=0)),
    (96, 1, 256, 32, [500, 64], 1, dict(causal=False, fp8=True)),
    # Few streams over a table far wider than the rows: 70 to 130 parts each.
    (16, 1, 64, 256, [20000], 8, dict(causal=True)),
    (16, 1, 128, 64, [16000, 5000], 8, dict(causal=True, fp8=True, dtype=0)),
    (16, 1, 256, 16, [9000], 9, dict(causal=True, softcap=20.0, dtype=0)),
    # Windows whose first tile holds whole pages behind them.
    (8, 2, 128, 16, [900, 470, 100], 64, dict(causal=True, window=(200, 0), dtype=0)),
    (8, 2, 128, 16, [900, 490], 64, dict(causal=True, window=(200, 0), fp8=True)),
    (8, 2, 64, 32, [870, 490], 64, dict(causal=True, window=(200, 0))),
    (8, 2, 256, 32, [870, 480], 64, dict(causal=False, window=(200, 30), fp8=True, dtype=0)),
]


def desc_plan(q, kc, bt, **kw):
    """(waves, workspace bytes) of the call's plan."""
    import pagedkv

    B, M, H, D = q.shape
    d = pagedkv.make_desc(batch=B, num_heads=H, num_heads_k=kc.shape[2], head_dim=D, page_size=kc.shape[1],
                          num_pages=kc.shape[0], block_table_stride=bt.shape[1], seqlen_q=M, **kw)
    return pagedkv.num_splits_for(d), pagedkv.workspace_size(d)


def prefill_workspace(waves, D):
    assert waves >= 4  # four a workgroup
    rows = waves // 4 * 2 * 128
    up = lambda x: (x + 255) // 256 * 256  # noqa: E731
    return up(rows * D * 4) + up(rows * 4 + waves // 4 * 16)


def hide(kc, vc, bt, lens, first, nan):
    """Copies with every slot that no query sees (positions below first[b], or past the row) filled with
    `nan`, and the pages that hold none let go, as an engine does behind a window: their table entries
    become -1, which the kernels read as page 0, itself made all `nan`."""
    kc, vc, bt = kc.copy(), vc.copy(), bt.copy()
    P = kc.shape[1]
    used = {int(bt[b, j]) for b, n in enumerate(lens) for j in range(first[b] // P, -(-max(n, 0) // P))}
    spare = next(i for i in range(kc.shape[0]) if i not in used)
    for c in (kc, vc):
        c[[0, spare]] = c[[spare, 0]]
    bt[bt == 0] = spare
    seen = np.zeros(kc.shape[:2], bool)
    for b, n in enumerate(lens):
        bt[b, :first[b] // P] = -1
        t = np.arange(first[b], max(n, 0))
        seen[bt[b, t // P], t % P] = True
    assert not seen[0].any()
    kc[~seen] = nan
    vc[~seen] = nan
    return kc, vc, bt


@pytest.mark.parametrize("case", range(len(CASES)))
def test_prefill_matches_oracle(case):
    import pagedkv

    torch = torch_mod()
    H, Hk, D, P, lens, M, opt = CASES[case]
    announce("prefill", CASES[case])
    rng = np.random.default_rng(9100 + case)
    dtype, fp8, B = opt.get("dtype", 1), opt.get("fp8", False), len(lens)
    window, leftpad = opt.get("window", (-1, -1)), opt.get("leftpad")
    blocks = B * Hk * -(-(M * H // Hk) // 32)
    stride = -(-12000 * 64 // blocks) // P + 1  # a table wide enough for the kernel to be chosen
    if window[0] >= 0:
        H, Hk, lens, B = H * 8, Hk * 8, lens * 8, B * 8  # a window bounds the work: more rows instead
        leftpad = None if leftpad is None else leftpad * 8
        stride = 1
    _, kc, vc, bt, sl = make_case(rng, B=B, H=H, Hk=Hk, D=D, P=P, seqlens=lens, dtype=dtype, stride=stride)
    q = rand_bits(rng, (B, M, H, D), dtype)
    scale = opt.get("scale", 1.0 / math.sqrt(D))
    slopes = rng.uniform(0.01, 0.3, size=(B, H)).astype(np.float32) if opt.get("alibi") else None
    cap = opt.get("softcap", 0.0)
    first = [0 if leftpad is None else leftpad[b] for b in range(B)]  # the first key some query of the row sees
    if window[0] >= 0:
        first = [max(f, n - M - window[0]) for f, n in zip(first, lens)]
    ks = vs = None
    kw = dict(causal=opt["causal"], window=window, alibi=slopes, lse=True, leftpad=None if leftpad is None else
              np.asarray(leftpad, np.int32), softcap=cap)
    if fp8:
        ks, vs = (rng.uniform(0.2, 2.0, Hk).astype(np.float32) for _ in range(2))
        kc, vc = fp8_cache(rng, kc.shape, ks), fp8_cache(rng, vc.shape, vs)
        want, want_lse = po.attn8_f64(q, kc, vc, bt, sl, scale, dtype, k_scale=ks, v_scale=vs, **kw)
    else:
        want, want_lse = po.attn_f64(q, kc, vc, bt, sl, scale, dtype, **kw)
    waves, need = desc_plan(q, kc, bt, dtype=dtype, causal=opt["causal"], window_size=window,
                            kv_dtype=pagedkv.PKV_KV_DTYPE_FP8_E4M3 if fp8 else 0)
    assert need == prefill_workspace(waves, D)
    lse = lse_buffer(B, H, M)

    def args(first):
        k, v, table = hide(kc, vc, bt, lens, first, 0x7F if fp8 else 0x7FC0 if dtype == 1 else 0x7E00)
        k, v = (to_dev8(k), to_dev8(v)) if fp8 else (to_dev(k, dtype), to_dev(v, dtype))
        return to_dev(q, dtype), k, v, i32(table), i32(sl), scale, 0

    more = dict(causal=opt["causal"], window_size=window, alibi_slopes=f32(slopes), k_scale=f32(ks), v_scale=f32(vs),
                softcap=cap, cache_leftpad=None if leftpad is None else i32(np.asarray(leftpad, np.int32)))
    out = pagedkv.decode(*args(first), softmax_lse=lse, **more)
    torch.cuda.synchronize()
    assert_close(out, want, dtype)
    assert_lse(lse, want_lse)
    # A workspace that only the decode kernels' plan fits (1,024 waves' and the streams' slots of 32
    # rows at most): that plan, within the same tolerance.  Those kernels read from the 16-token tile of
    # the first key on, behind a window too.
    if need - 256 >= (1024 + B * Hk * -(-(M * H // Hk) // 32)) * 32 * (D + 1) * 4 + 512:
        first = first if leftpad is not None else [f // 16 * 16 for f in first]
        small = pagedkv.decode(*args(first), workspace=torch.empty(need - 256, dtype=torch.uint8, device="cuda"), **more)
        torch.cuda.synchronize()
        assert_close(small, want, dtype)


def test_prefill_many_ragged_rows():
    """More rows than threads in a workgroup, one to three row blocks each, rows without tokens
    among them: shares cross rows, blocks and KV heads."""
    import pagedkv

    torch = torch_mod()
    announce("prefill-ragged")
    rng = np.random.default_rng(9200)
    B, H, Hk, D, P, M, dtype = 300, 4, 2, 128, 16, 70, 1
    lens = rng.integers(0, 400, size=B).astype(np.int32)
    lens[:3] = (0, 1, 399)
    _, kc, vc, bt, sl = make_case(rng, B=B, H=H, Hk=Hk, D=D, P=P, seqlens=lens, dtype=dtype)
    q = rand_bits(rng, (B, M, H, D), dtype)
    want = po.attn_f64(q, kc, vc, bt, sl, 0.09, dtype, causal=True)
    waves, need = desc_plan(q, kc, bt, dtype=dtype, causal=True)
    assert need == prefill_workspace(waves, D)
    out = pagedkv.decode(to_dev(q, dtype), to_dev(kc, dtype), to_dev(vc, dtype), i32(bt), i32(sl), 0.09, 0,
                         causal=True)
    torch.cuda.synchronize()
    assert_close(out, want, dtype)


def test_prefill_at_its_limit_of_row_blocks():
    """1,024 rows of two row blocks: as many entries as the plan in the LDS holds."""
    import pagedkv

    torch = torch_mod()
    announce("prefill-entries")
    rng = np.random.default_rng(9250)
    B, H, Hk, D, P, M, dtype = 1024, 4, 1, 64, 16, 33, 0
    lens = rng.integers(0, 129, size=B).astype(np.int32)
    _, kc, vc, bt, sl = make_case(rng, B=B, H=H, Hk=Hk, D=D, P=P, seqlens=lens, dtype=dtype, stride=8)
    q = rand_bits(rng, (B, M, H, D), dtype)
    want = po.attn_f64(q, kc, vc, bt, sl, 0.12, dtype, causal=True)
    waves, need = desc_plan(q, kc, bt, dtype=dtype, causal=True)
    assert need == prefill_workspace(waves, D)
    out = pagedkv.decode(to_dev(q, dtype), to_dev(kc, dtype), to_dev(vc, dtype), i32(bt), i32(sl), 0.12, 0,
                         causal=True)
    torch.cuda.synchronize()
    assert_close(out, want, dtype)


def test_prefill_under_graph_replays():
    """A captured appending prefill chunk, replayed several times with eager work in between."""
    import pagedkv

    torch = torch_mod()
    announce("prefill-graph")
    rng = np.random.default_rng(9300)
    B, H, Hk, D, P, M, dtype = 2, 32, 8, 128, 16, 96, 1
    _, kc, vc, bt, sl = make_case(rng, B=B, H=H, Hk=Hk, D=D, P=P, seqlens=[1500, 700], dtype=dtype, stride=200)
    q, kn, vn = rand_bits(rng, (B, M, H, D), dtype), *(rand_bits(rng, (B, M, Hk, D), dtype) for _ in range(2))
    waves, need = desc_plan(q, kc, bt, dtype=dtype, causal=True)
    assert need == prefill_workspace(waves, D)
    k2, v2 = po.append_kv(kc, vc, bt, np.asarray(sl) - M, kn, vn)
    exact = po.attn_f64(q, k2, v2, bt, sl, 0.09, dtype, causal=True)
    q, kn, vn, kd, vd = (to_dev(t, dtype) for t in (q, kn, vn, kc, vc))
    table, lens = i32(bt), i32(np.asarray(sl) - M)

    def call():
        return pagedkv.decode(q, kd, vd, table, lens, 0.09, 0, k_new=kn, v_new=vn, causal=True)

    want = call().clone()
    torch.cuda.synchronize()
    assert_close(want, exact, dtype)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        got = call()
    for _ in range(4):
        got.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)
        assert torch.equal(call(), want)


@pytest.mark.parametrize("D,fp8", [(128, False), (64, True)])
def test_long_verify_step_appends_then_attends(D, fp8):
    """A verify step past the fold's work: the new tokens are in the caches bit for bit, the output is
    the oracle's over the longer rows."""
    import pagedkv

    torch = torch_mod()
    announce("prefill-verify", D, fp8)
    rng = np.random.default_rng(9400 + D)
    B, H, Hk, P, M, dtype = 3, 32, 2, 16, 8, 1
    stride = -(-13000 * 64 // (B * Hk * 4)) // P + 1
    total = np.array([900, 72, 8], np.int32)
    _, kc, vc, bt, _ = make_case(rng, B=B, H=H, Hk=Hk, D=D, P=P, seqlens=total, dtype=dtype, stride=stride)
    q = rand_bits(rng, (B, M, H, D), dtype)
    kn, vn = (rand_bits(rng, (B, M, Hk, D), dtype) for _ in range(2))
    old = total - M
    ks = vs = None
    if fp8:
        ks, vs = (rng.uniform(0.2, 2.0, Hk).astype(np.float32) for _ in range(2))
        kc, vc = fp8_cache(rng, kc.shape, ks), fp8_cache(rng, vc.shape, vs)
        k2, v2 = po.append_kv(kc, vc, bt, old, po.quantize_e4m3(kn, dtype, ks),
                              po.quantize_e4m3(vn, dtype, vs))
        want = po.attn8_f64(q, k2, v2, bt, total, 0.1, dtype, k_scale=ks, v_scale=vs, causal=True)
        kd, vd = to_dev8(kc), to_dev8(vc)
    else:
        k2, v2 = po.append_kv(kc, vc, bt, old, kn, vn)
        want = po.attn_f64(q, k2, v2, bt, total, 0.1, dtype, causal=True)
        kd, vd = to_dev(kc, dtype), to_dev(vc, dtype)
    desc = pagedkv.make_desc(batch=B, num_heads=H, num_heads_k=Hk, head_dim=D, page_size=P, num_pages=kc.shape[0],
                             block_table_stride=stride, seqlen_q=M, dtype=dtype, causal=True,
                             kv_dtype=pagedkv.PKV_KV_DTYPE_FP8_E4M3 if fp8 else 0)
    assert pagedkv.append_folds(desc, 0, M) is False
    assert pagedkv.workspace_size(desc) == prefill_workspace(pagedkv.num_splits_for(desc), D)
    out = pagedkv.decode(to_dev(q, dtype), kd, vd, i32(bt), i32(old), 0.1, 0, k_new=to_dev(kn, dtype),
                         v_new=to_dev(vn, dtype), causal=True, k_scale=f32(ks), v_scale=f32(vs))
    torch.cuda.synchronize()
    assert_close(out, want, dtype)
    for got, exact in ((kd, k2), (vd, v2)):
        np.testing.assert_array_equal(from_dev8(got) if fp8 else from_dev(got), exact)


@pytest.mark.parametrize("D,M,lens,dtype", [
    (128, 40, [2100, 1700], 1),          # few streams: cut into many parts
    (64, 40, [2100, 1700], 0),
    (256, 40, [2100, 1700], 1),
    (128, 70, [1 + 7 * (i % 9) for i in range(64)], 0),  # rows of one tile: whole streams
])
def test_nan_query_rows_stay_nan(D, M, lens, dtype):
    """A query row that holds a NaN gives NaN, whether its stream is cut or not, and no other row
    does."""
    import pagedkv

    torch = torch_mod()
    announce("prefill-nan", D, M, len(lens), dtype)
    rng = np.random.default_rng(9500 + D + M)
    B, H, Hk, P = len(lens), 16, 4, 16
    stride = -(-13000 * 64 // (B * Hk * -(-(M * H // Hk) // 32))) // P + 1
    _, kc, vc, bt, sl = make_case(rng, B=B, H=H, Hk=Hk, D=D, P=P, seqlens=lens, dtype=dtype, stride=stride)
    q = rand_bits(rng, (B, M, H, D), dtype)
    nan = rng.random((B, M, H)) < 0.02
    nan[0, 0, 0] = nan[-1, -1, -1] = True
    want, want_lse = po.attn_f64(q, kc, vc, bt, sl, 0.1, dtype, lse=True)
    q[nan, 5] = 0x7FC0 if dtype == 1 else 0x7E00
    waves, need = desc_plan(q, kc, bt, dtype=dtype)
    assert need == prefill_workspace(waves, D)
    lse = lse_buffer(B, H, M)
    out = pagedkv.decode(to_dev(q, dtype), to_dev(kc, dtype), to_dev(vc, dtype), i32(bt), i32(sl), 0.1, 0,
                         softmax_lse=lse)
    torch.cuda.synchronize()
    got = po.bits_to_f32(from_dev(out), dtype)
    np.testing.assert_array_equal(np.isnan(got), np.broadcast_to(nan[..., None], got.shape))
    excess = np.abs(got - want) - (TOL[dtype] + REL[dtype] * np.abs(want))
    assert np.max(excess[~nan]) < 0
    lse_nan = nan.transpose(0, 2, 1)
    want_lse[lse_nan] = np.inf  # as the decode kernels write it
    assert_lse(lse, want_lse)


@pytest.mark.parametrize("H,Hk,D,B,M,bound,longest,dtype,opt", [
    (32, 8, 256, 32, 40, 511, 128, 1, dict(causal=True)),
    (128, 32, 64, 180, 5, 1024, 70, 0, dict(causal=True)),                    # 20 query rows per KV head
    (128, 32, 64, 180, 5, 1024, 70, 1, dict(causal=True, window=(50, 0))),
    (64, 32, 128, 110, 17, 1024, 40, 1, dict(causal=False, fp8=True)),         # 34 rows
])
def test_workspace_sized_for_longer_rows(H, Hk, D, B, M, bound, longest, dtype, opt):
    """A workspace sized for a large prefill, given to a call of short rows or few query tokens whose
    decode plan needs more: the call takes the prefill kernel instead of being refused."""
    import pagedkv

    torch = torch_mod()
    announce("prefill-small-workspace", H, Hk, D, B, M, bound, longest, dtype, opt)
    rng = np.random.default_rng(9600 + D + M)
    P, fp8, causal, window = 16, opt.get("fp8", False), opt["causal"], opt.get("window", (-1, -1))
    lens = rng.integers(0, longest + 1, size=B).astype(np.int32)
    lens[:3] = (0, 1, longest)
    _, kc, vc, bt, sl = make_case(rng, B=B, H=H, Hk=Hk, D=D, P=P, seqlens=lens, dtype=dtype, stride=bound // P)
    q = rand_bits(rng, (B, M, H, D), dtype)
    kv_dtype = pagedkv.PKV_KV_DTYPE_FP8_E4M3 if fp8 else 0
    at_hand = desc_plan(rand_bits(rng, (B, max(M, 40), 1, D), dtype).repeat(H, axis=2), kc, bt, dtype=dtype, causal=True,
                        max_seqlen=bound, kv_dtype=kv_dtype)[1]
    waves, need = desc_plan(q, kc, bt, dtype=dtype, causal=causal, window_size=window, max_seqlen=longest,
                            kv_dtype=kv_dtype)
    assert need > at_hand
    ks = vs = None
    if fp8:
        ks, vs = (rng.uniform(0.2, 2.0, Hk).astype(np.float32) for _ in range(2))
        kc, vc = fp8_cache(rng, kc.shape, ks), fp8_cache(rng, vc.shape, vs)
        want, want_lse = po.attn8_f64(q, kc, vc, bt, sl, 0.1, dtype, k_scale=ks, v_scale=vs, causal=causal,
                                      window=window, lse=True)
    else:
        want, want_lse = po.attn_f64(q, kc, vc, bt, sl, 0.1, dtype, causal=causal, window=window, lse=True)
    lse = lse_buffer(B, H, M)
    out = pagedkv.decode(to_dev(q, dtype), to_dev8(kc) if fp8 else to_dev(kc, dtype),
                         to_dev8(vc) if fp8 else to_dev(vc, dtype), i32(bt), i32(sl), 0.1, 0, causal=causal,
                         window_size=window, max_seqlen=longest, k_scale=f32(ks), v_scale=f32(vs), softmax_lse=lse,
                         workspace=torch.empty(at_hand, dtype=torch.uint8, device="cuda"))
    torch.cuda.synchronize()
    assert_close(out, want, dtype)
    assert_lse(lse, want_lse)


def test_misaligned_workspace_where_none_is_needed():
    """Rows bounded by a window: the decode kernels' plan is the single pass, so a workspace that the
    prefill kernel cannot use does not stop the call."""
    import pagedkv

    torch = torch_mod()
    announce("prefill-misaligned-workspace")
    rng = np.random.default_rng(9650)
    B, H, Hk, D, P, M, dtype, window = 16, 64, 16, 128, 16, 64, 1, (200, 0)
    _, kc, vc, bt, sl = make_case(rng, B=B, H=H, Hk=Hk, D=D, P=P, seqlens=[900, 490] * 8, dtype=dtype)
    q = rand_bits(rng, (B, M, H, D), dtype)
    waves, need = desc_plan(q, kc, bt, dtype=dtype, causal=True, window_size=window)
    assert need == prefill_workspace(waves, D)
    want = po.attn_f64(q, kc, vc, bt, sl, 0.1, dtype, causal=True, window=window)
    out = pagedkv.decode(to_dev(q, dtype), to_dev(kc, dtype), to_dev(vc, dtype), i32(bt), i32(sl), 0.1, 0,
                         causal=True, window_size=window,
                         workspace=torch.empty(need + 16, dtype=torch.uint8, device="cuda")[8:])
    torch.cuda.synchronize()
    assert_close(out, want, dtype)


def test_verify_step_folds_in_a_workspace_for_the_fold():
    """A verify step with the prefill kernel's work, given a workspace that holds only the folded
    plan's partials: the oracle's output, the new tokens in the caches bit for bit."""
    import pagedkv

    torch = torch_mod()
    announce("prefill-verify-fold-workspace")
    rng = np.random.default_rng(9700)
    B, H, Hk, D, P, M, dtype = 3, 32, 2, 128, 16, 8, 1
    stride = -(-13000 * 64 // (B * Hk * 4)) // P + 1
    total = np.array([900, 72, 8], np.int32)
    _, kc, vc, bt, _ = make_case(rng, B=B, H=H, Hk=Hk, D=D, P=P, seqlens=total, dtype=dtype, stride=stride)
    q = rand_bits(rng, (B, M, H, D), dtype)
    kn, vn = (rand_bits(rng, (B, M, Hk, D), dtype) for _ in range(2))
    k2, v2 = po.append_kv(kc, vc, bt, total - M, kn, vn)
    want = po.attn_f64(q, k2, v2, bt, total, 0.1, dtype, causal=True)
    rows = (1024 + B * Hk * 4) * 32
    workspace = torch.empty(256 + rows * D * 4 + rows * 4, dtype=torch.uint8, device="cuda")
    kd, vd = to_dev(kc, dtype), to_dev(vc, dtype)
    out = pagedkv.decode(to_dev(q, dtype), kd, vd, i32(bt), i32(total - M), 0.1, 0, k_new=to_dev(kn, dtype),
                         v_new=to_dev(vn, dtype), causal=True, workspace=workspace)
    torch.cuda.synchronize()
    assert_close(out, want, dtype)
    for got, exact in ((kd, k2), (vd, v2)):
        np.testing.assert_array_equal(from_dev(got), exact)
