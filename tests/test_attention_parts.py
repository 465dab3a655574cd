"""Attention over key parts read where they lie (hn_segment_attention, hy_nomas/model.py:199-223): the V^T packing, the
segments' masked last tiles, the groups' gathered rows, against float32 softmax attention over the joined keys and
against the one-call-per-group form; and on the CPU, which plans take it and what its entry point refuses."""
import ctypes

import pytest
import torch

from conftest import seeded
from test_attention_gpu import Plan, ref_attention, rel


def operands(dev, b, h, lv, lt, lh, seed, head_major=False):
    g = seeded(seed)

    def make(n, batch=b):
        if head_major:
            return torch.randn(batch, h, n, 128, generator=g).to(torch.bfloat16).to(dev).transpose(1, 2)
        return torch.randn(batch, n, h, 128, generator=g).to(torch.bfloat16).to(dev)

    q, k, v = make(lv + lt), make(lv + lt), make(lv + lt)
    return q, k, v, (make(lh, 1), make(lh, 1)) if lh else None


def split_plan(dev, lv, lt, n):
    tok, txt = torch.arange(lv, device=dev).tensor_split(n), torch.arange(lt, device=dev).tensor_split(n)
    return Plan(lv, [(torch.cat([a, lv + t]), t) for a, t in zip(tok, txt)])


def per_group(q, k, v, hist, plan):
    lv, ref = plan.video_tokens, torch.full(q.shape, float("nan"), device=q.device)
    hk, hv = (t.expand(q.shape[0], -1, -1, -1) for t in hist) if hist else (k[:, :0], v[:, :0])
    for qi, ti in plan.groups:
        keys, vals = (torch.cat([x, t[:, :lv], t[:, lv + ti]], dim=1) for x, t in ((hk, k), (hv, v)))
        ref[:, qi] = ref_attention(q[:, qi], keys, vals)
    return ref


# lengths around the 64-key tile, the 128-query block and the workgroup's 32-query waves; no history, no text keys
# for a group, more groups than text tokens; token-major and head-major operands; a batch of two over one history
@pytest.mark.gpu
@pytest.mark.parametrize("b,h,lv,lt,lh,n,head_major", [
    (1, 2, 63, 7, 0, 2, False), (1, 3, 64, 64, 64, 1, False), (2, 2, 129, 5, 65, 3, False), (1, 1, 1, 1, 1, 1, True),
    (2, 3, 300, 130, 191, 4, True), (1, 2, 200, 3, 127, 5, False), (1, 2, 130, 0, 70, 2, False),
    (1, 1, 150, 70, 33, 70, False), (1, 2, 0, 40, 0, 2, False), (1, 2, 0, 33, 70, 2, False),
    # few queries over many keys: several workgroups share a query block's keys, with ranges that start and end in
    # the history, the video keys and the text keys
    (1, 2, 129, 40, 1900, 3, False), (2, 1, 40, 200, 511, 2, True), (1, 1, 900, 1, 0, 1, False),
    (1, 3, 20, 600, 64, 1, False),
    # more query blocks than a round of workgroups (512 on 256 compute units): only those past it are split
    (1, 24, 2700, 100, 300, 2, False), (2, 20, 1700, 3, 0, 1, True)])
def test_groups_against_float32(dev, b, h, lv, lt, lh, n, head_major):
    from hy_nomas import attention

    print(f"groups b={b} h={h} lv={lv} lt={lt} lh={lh} n={n} head_major={head_major}", flush=True)
    q, k, v, hist = operands(dev, b, h, lv, lt, lh, lv + lt + lh, head_major)
    plan = split_plan(dev, lv, lt, n)
    got = attention.segment_attention(q, k, v, hist, plan, backend="hip")
    assert got.stride() == torch.empty_like(q).stride()
    fro, mx = rel(got, per_group(q, k, v, hist, plan))
    assert fro < 1e-2 and mx < 3e-2, (fro, mx)  # bf16 operands, probabilities and result, as test_attention_gpu


@pytest.mark.gpu
@pytest.mark.parametrize("lq,lh", [(1, 1), (64, 63), (65, 64), (200, 129)])
def test_history_without_groups(dev, lq, lh):
    from hy_nomas import attention

    q, k, v, hist = operands(dev, 1, 2, lq, 0, lh, lq * 3 + lh)
    got = attention.segment_attention(q, k, v, hist, None, backend="hip")
    ref = ref_attention(q, torch.cat([hist[0], k], dim=1), torch.cat([hist[1], v], dim=1))
    fro, mx = rel(got, ref)
    assert fro < 1e-2 and mx < 3e-2, (fro, mx)


@pytest.mark.gpu
def test_overlapping_negative_and_repeated_rows(dev):
    """A row in two groups takes the later group's result; negative rows count from the end; a group may name a row
    twice.  Rows in no group are left alone."""
    from hy_nomas import attention

    lv, lt = 150, 20
    q, k, v, hist = operands(dev, 1, 2, lv, lt, 40, 5)
    at = lambda *x: torch.tensor(x, device=dev)  # noqa: E731
    plan = Plan(lv, [(torch.arange(0, 100, device=dev), at(0, 1)), (torch.arange(60, 140, device=dev), at(5, -1, 5)),
                     (at(-1, 3, 3), at(7))])
    out = torch.zeros_like(q)
    attention._segment(q, k, v, hist, plan, "hip", out=out)
    ref = per_group(q, k, v, hist, plan)
    named = ~ref.isnan().any(-1).any(-1)[0]
    fro, mx = rel(out[:, named], ref[:, named])
    assert fro < 1e-2 and mx < 3e-2, (fro, mx)
    assert (out[:, ~named] == 0).all() and (~named).sum() == lv + lt - 141


@pytest.mark.gpu
@pytest.mark.parametrize("lk", [1, 15, 64, 100, 321])
def test_packed_values_equal_the_torch_layout(dev, lk):
    """One part with no groups against the kernel on `transpose_values`: the same products, bit for bit."""
    from hy_nomas import attention

    q, k, v, _ = operands(dev, 2, 2, lk, 0, 0, lk)
    got = attention.attention(q, k, v, backend="hip")
    assert torch.equal(got, attention.attention_hip(q, k, attention.transpose_values(v.transpose(1, 2)), lk))


def test_which_plans_take_the_rows():
    from hy_nomas import attention

    q = torch.empty(1, 12, 1, 128, dtype=torch.bfloat16)
    good = (torch.arange(10), torch.arange(2))

    def ok(groups, lv=10, hist=None, out=q):
        return attention._groups_ok(q, q, q, hist, Plan(lv, groups), out)

    assert ok([good]) and ok((good, good)) and ok([good], lv=0)
    assert not ok([]) and not ok(iter([good])) and not ok([good], lv=13) and not ok([good], lv=-1)
    for bad in (torch.arange(12) > 3, torch.arange(10, dtype=torch.int32), [0, 1], slice(0, 3), torch.zeros(2, 2).long()):
        assert not ok([(bad, good[1])]) and not ok([good, (good[0], bad)])
    assert not ok([(good[0], good[1][:0])], lv=0)  # no keys: the general form refuses it
    assert ok([(good[0], good[1][:0])], lv=0, hist=(q, q))
    assert not ok([good], out=torch.empty(1, 12, 128, 1, dtype=torch.bfloat16).transpose(2, 3))


def test_argument_validation_without_a_gpu():
    from hy_nomas import _lib

    lib, p = _lib.lib(), 4096  # never dereferenced: every call below is refused on the host

    def call(parts, groups=(), b=1, h=1, lq=10, d=128, scale=1.0, ws=p, nbytes=1 << 40, rows=p):
        pt, gr = _lib.int64s(parts), _lib.int64s(groups) if groups else None
        text = _lib.int64s([p, 0, 128, 128] * 2)
        return lib.hn_segment_attention(p, 0, 128, 128, pt, len(parts) // 9, text, gr, len(groups) // 4, rows, 0, p, 0, 128,
                                        128, b, h, lq, d, scale, ws, nbytes, None)

    part = [p, 0, 128, 128, p, 0, 128, 128, 64]
    for bad in (call(part, d=64), call([]), call(part * 3), call(part[:8] + [0]), call(part, scale=0.0),
                call([p + 8] + part[1:]), call(part[:3] + [4] + part[4:]), call(part[:7] + [0, 64]),
                call(part, nbytes=100), call(part, ws=p + 16), call(part, h=70000), call(part, groups=[0, 4, 0, 1], rows=None),
                call(part[:8] + [0], groups=[0, 4, 0, 0]), call(part, groups=[0, 1, 0, 0] * 65),
                call(part[:8] + [(1 << 22) + 1])):
        assert bad != 0 and lib.hn_last_error()
    assert lib.hn_segment_attention_workspace_bytes(_lib.int64s(part), 1, None, 0, 1, 1, 10) == 128 * 64 * 2
    assert lib.hn_segment_attention_workspace_bytes(_lib.int64s(part), 3, None, 0, 1, 1, 10) == -1
    assert ctypes.sizeof(_lib.int64s(part)) == 72


# units (of 128 queries) x keys: the keys walked by one workgroup, and split into ranges that begin inside the mask
@pytest.mark.gpu
@pytest.mark.parametrize("h,lq,lk,masked", [(1, 129, 100, (0, 64)), (1, 129, 2000, (64, 1900)), (1, 129, 2000, (0, 1900)),
                                            (2, 40, 1500, (700, 1500)), (24, 2700, 1500, (64, 1500))])
def test_tiles_whose_scores_are_all_minus_infinity(dev, h, lq, lk, masked):
    """Keys hidden from every other query by a product beyond the floats' range: whole tiles score -inf for some of a
    wave's queries and not for others, first in a range of keys or later.  They take no weight."""
    from hy_nomas import attention

    q, k, v, _ = operands(dev, 1, h, max(lq, lk), 0, 0, lq + lk)
    q, k, v = q[:, :lq].clone(), k[:, :lk].clone(), v[:, :lk]
    q[..., 0] = 0
    q[:, ::2, :, 0] = 4
    k[:, masked[0]:masked[1], :, 0] = torch.finfo(torch.bfloat16).min
    ref = ref_attention(q, k, v)
    assert torch.isfinite(ref).all()
    got = attention.attention(q, k, v, backend="hip")
    assert torch.isfinite(got.float()).all()
    fro, mx = rel(got, ref)
    assert fro < 1e-2 and mx < 3e-2, (fro, mx)


def off16(t, by=1):
    """t's values in a contiguous tensor that starts `by` elements past a 16-byte boundary."""
    flat = torch.empty(t.numel() + by, dtype=t.dtype, device=t.device)[by:]
    return flat.view(t.shape).copy_(t)


def test_rows16_copies_what_contiguous_leaves():
    """A contiguous tensor off a 16-byte boundary, and one whose size-1 dims have odd strides, are copied too."""
    from hy_nomas import attention

    t = torch.randn(1, 6, 2, 128).to(torch.bfloat16)
    odd = torch.empty(3000, dtype=torch.bfloat16).as_strided((1, 6, 2, 128), (1537, 256, 128, 1)).copy_(t)
    for x in (off16(t), off16(t, 4), odd, t[..., ::2].repeat_interleave(2, -1).transpose(2, 3).contiguous().transpose(2, 3)):
        got = attention._rows16(x)
        assert torch.equal(got, x) and got.stride(-1) == 1
        assert got.data_ptr() % 16 == 0 and all(st % 8 == 0 for st in got.stride()[:-1])
    assert attention._rows16(t) is t and attention._rows16(t[:, 1:]).data_ptr() == t[:, 1:].data_ptr()


@pytest.mark.gpu
def test_operands_off_the_16_byte_boundary(dev):
    """Queries, keys, values and history that start anywhere, with and without groups: the aligned tensors' result."""
    from hy_nomas import attention

    q, k, v, hist = operands(dev, 1, 2, 130, 20, 70, 9)
    for plan in (None, split_plan(dev, 130, 20, 2)):
        want = attention.segment_attention(q, k, v, hist, plan, backend="hip")
        got = attention.segment_attention(off16(q), off16(k, 2), off16(v), tuple(map(off16, hist)), plan, backend="hip")
        assert torch.equal(got, want)
    assert torch.equal(attention.attention(off16(q), off16(k), off16(v), backend="hip"),
                       attention.attention(q, k, v, backend="hip"))


@pytest.mark.gpu
def test_groups_without_queries(dev):
    """Plans whose groups, all of them or those of a whole launch (past the 64th), name no query or text rows."""
    from hy_nomas import attention

    q, k, v, hist = operands(dev, 1, 2, 70, 6, 40, 11)
    none, text = torch.arange(0, device=dev), torch.arange(2, device=dev)
    rows = torch.arange(50, device=dev)
    for groups in ([(none, none)], [(none, text)], [(rows, text)] + [(none, none)] * 64, [(none, none)] * 70 + [(rows, text)]):
        out = torch.zeros_like(q)
        attention._segment(q, k, v, hist, Plan(70, groups), "hip", out=out)
        assert (out[:, 50:] == 0).all()
        if any(t.numel() for t, _ in groups):
            fro, mx = rel(out[:, :50], per_group(q, k, v, hist, Plan(70, [(rows, text)]))[:, :50])
            assert fro < 1e-2 and mx < 3e-2, (fro, mx)
        else:
            assert (out == 0).all()


# few queries over many keys (split), and several blocks over few (not)
@pytest.mark.gpu
@pytest.mark.parametrize("lv,lt,lh", [(129, 40, 1900), (300, 130, 60)])
def test_non_finite_operands(dev, lv, lt, lh):
    """Infinite and NaN values reach the outputs that weigh them, a NaN query only its own row, and a key of infinite
    scores takes no weight (-inf) or makes its query NaN (+inf), through the packed values and the joined partials."""
    from hy_nomas import attention

    q, k, v, hist = operands(dev, 1, 2, lv, lt, lh, 17)
    plan = split_plan(dev, lv, lt, 2)
    hist[1][0, 3, 0, 5], v[0, 70, 0, 6], v[0, lv + 1, 1, 7] = float("inf"), float("-inf"), float("nan")
    q[0, 9, 1, 0], k[0, 2, 1, 3] = float("nan"), float("inf")
    got, ref = attention.segment_attention(q, k, v, hist, plan, backend="hip").float(), per_group(q, k, v, hist, plan)
    assert torch.equal(got.isnan(), ref.isnan()) and ref.isnan().any() and (~ref.isnan()).any()
    assert torch.equal(got.isinf(), ref.isinf()) and torch.equal(got[got.isinf()], ref[ref.isinf()])
    fin = ref.isfinite()
    fro, mx = rel(got[fin], ref[fin])
    assert fro < 1e-2 and mx < 3e-2, (fro, mx)


@pytest.mark.gpu
@pytest.mark.parametrize("h,lv,lt,lh", [(2, 129, 40, 1900), (24, 2700, 100, 300)])
def test_repeated_calls_give_the_same_bits(dev, h, lv, lt, lh):
    from hy_nomas import attention

    q, k, v, hist = operands(dev, 1, h, lv, lt, lh, 23)
    for plan in (None, split_plan(dev, lv, lt, 3)):
        first = attention.segment_attention(q, k, v, hist, plan, backend="hip")
        for _ in range(3):
            assert torch.equal(attention.segment_attention(q, k, v, hist, plan, backend="hip"), first)


@pytest.mark.gpu
@pytest.mark.parametrize("groups", [0, 3])
def test_segment_attention_under_graph_capture(dev, groups):
    """One captured call replayed on fresh inputs, with eager work and synchronizations between the replays."""
    from hy_nomas import attention

    lv, lt, lh = 129, 40, 1900
    q, k, v, hist = operands(dev, 1, 2, lv, lt, lh, 29)
    plan = split_plan(dev, lv, lt, groups) if groups else None

    def call():
        return attention.segment_attention(q, k, v, hist, plan, backend="hip")

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    torch.cuda.synchronize()
    for replay in range(3):
        for t, new in zip((q, k, v, *hist), (*(x := operands(dev, 1, 2, lv, lt, lh, 31 + replay))[:3], *x[3])):
            t.copy_(new)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, call()), replay


@pytest.mark.gpu
@pytest.mark.parametrize("b,h,lq,lk", [(1, 1, 1, 1), (2, 3, 200, 130), (1, 2, 129, 2000), (1, 24, 2700, 400)])
def test_entry_point_without_a_workspace(dev, b, h, lq, lk):
    """hn_attention, whose query blocks are never split, against float32."""
    from hy_nomas import _lib, attention

    q, k, v, _ = operands(dev, b, h, max(lq, lk), 0, 0, lq * lk)
    q, k, v, out = q[:, :lq], k[:, :lk], v[:, :lk], torch.empty(b, lq, h, 128, dtype=torch.bfloat16, device=dev)
    vt = attention.transpose_values(v.transpose(1, 2))
    _lib.call("hn_attention", *attention._operand(q), *attention._operand(k), vt.data_ptr(), *vt.stride()[:3],
              *attention._operand(out), b, h, lq, lk, 128, 128 ** -0.5, _lib.stream(q))
    fro, mx = rel(out, ref_attention(q, k, v))
    assert fro < 1e-2 and mx < 3e-2, (fro, mx)
