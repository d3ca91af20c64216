"""The block under torch.compile, traced on the CPU with fake device tensors: every
op is opaque (``ops``), so a denoising pass is one graph, as the reference's
compiled pre/post functions are (nomas_compile_prepost.py:14-99)."""
import pytest

from conftest import pkg_module

torch = pytest.importorskip("torch")


@pytest.fixture()
def traced(monkeypatch):
    """(block, inputs, graphs(fn, *args)) with every tensor fake and on "cuda"."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    db, dl, kvc = pkg_module("dit_block"), pkg_module("dit_fp8_linear"), pkg_module("fp8_kv_cache")
    # quantize_weight reads values (its finiteness check), which fake tensors lack
    monkeypatch.setattr(dl, "quantize_weight", lambda w: (
        torch.empty(w.shape, dtype=torch.float8_e4m3fn, device=w.device),
        torch.empty(w.shape[0], dtype=torch.float32, device=w.device)))
    L, Lt, hidden, heads = 132, 24, 512, 4

    def bf(*shape):
        return torch.empty(*shape, dtype=torch.bfloat16, device="cuda")

    with FakeTensorMode(allow_non_fake_inputs=True), torch.no_grad():
        blk = db.FP8DiTBlock(hidden, heads, device="cuda", text=True)
        rope = torch.empty(L, 128, device="cuda"), torch.empty(L, 128, device="cuda")
        cache = kvc.make_fp8_kv_block(1, 400, heads, 128, device="cuda")
        masks = dict(text_mask=torch.ones(1, Lt, dtype=torch.bool, device="cuda"),
                     cache_mask=torch.ones(1, 400, dtype=torch.bool, device="cuda"))
        x = dict(img=bf(1, L, hidden), txt=bf(1, Lt, hidden), vec=bf(1, hidden), rope=rope, cache=cache, masks=masks)

        def graphs(fn, *args):
            seen = []

            def backend(gm, example):
                seen.append(gm)
                return gm.forward
            torch._dynamo.reset()
            torch.compile(fn, backend=backend, fullgraph=True)(*args)
            return len(seen)
        yield blk, x, graphs
    torch._dynamo.reset()


def test_block_is_one_graph(traced):
    blk, x, graphs = traced
    assert graphs(lambda i, v: blk(i, v, *x["rope"], x["cache"], 132), x["img"], x["vec"]) == 1


def test_block_with_text_is_one_graph(traced):
    blk, x, graphs = traced

    def call(i, t, v):
        return blk(i, v, *x["rope"], x["cache"], 132, txt=t, vec_txt=v, **x["masks"])
    assert graphs(call, x["img"], x["txt"], x["vec"]) == 1


def test_block_halves_and_seam_are_one_graph_each(traced):
    blk, x, graphs = traced
    ca = pkg_module("cache_attention")
    assert graphs(lambda i, v: blk.pre_attention(i, v, *x["rope"]), x["img"], x["vec"]) == 1
    assert graphs(lambda t, v: blk.pre_attention_txt(t, v), x["txt"], x["vec"]) == 1
    parts = [torch.empty(1, 512, dtype=torch.bfloat16, device="cuda") for _ in range(6)]
    assert graphs(lambda i, a: blk.post_attention(i, a, parts), x["img"], torch.empty_like(x["img"])) == 1
    # QKV views, as pre_attention returns them
    img = torch.empty(1, 132, 3, 4, 128, dtype=torch.bfloat16, device="cuda").unbind(2)
    txt = torch.empty(1, 24, 3, 4, 128, dtype=torch.bfloat16, device="cuda").unbind(2)

    def seam(iq, ik, iv, tq, tk, tv):
        return ca.causal_attention_with_cache_mp((iq, tq), (ik, tk), (iv, tv), x["cache"], 132, "flash3",
                                                 x["masks"]["text_mask"], False, True, x["masks"]["cache_mask"])
    assert graphs(seam, *img, *txt) == 1


def test_write_verdict_under_compile_is_read_at_once():
    """A compiled write pass raises on its status word without pinned memory or events
    (neither exists in this process, and inductor traces neither)."""
    kvc = pkg_module("fp8_kv_cache")

    def call(status, x):
        refused = kvc.read_flag_later(status)
        y = x + 1
        refused()
        return y
    torch._dynamo.reset()
    compiled = torch.compile(call, backend="eager")
    assert torch.equal(compiled(torch.zeros(1, dtype=torch.int32), torch.ones(2)), torch.full((2,), 2.0))
    with pytest.raises(ValueError, match="non-finite"):
        compiled(torch.ones(1, dtype=torch.int32), torch.ones(2))
    torch._dynamo.reset()


def test_write_verdict_on_a_capturing_stream_is_read_at_once(monkeypatch):
    """No pinned memory and no event there: the plain read, which a capture refuses."""
    kvc = pkg_module("fp8_kv_cache")
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    kvc.read_flag_later(torch.zeros(1, dtype=torch.int32))()
    with pytest.raises(ValueError, match="non-finite"):
        kvc.read_flag_later(torch.ones(1, dtype=torch.int32))
