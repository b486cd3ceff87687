"""The native encoder loop against the same model's modules: token counts at the edges of its 16-row tiles and on both sides
of its own products, packed and full batches, and what makes it step aside."""
import copy
import ctypes as C
import threading

import pytest
import torch
from torch.utils.flop_counter import FlopCounterMode
from transformers import DebertaV2Config
from transformers.models.deberta_v2.modeling_deberta_v2 import DebertaV2Model

from golden_inputs import fill_params
from turbodeberta_amd import _lib
from turbodeberta_amd.model import FlashDebertaV2Model, _native_plan, declare_right_padded, patch_model

pytestmark = pytest.mark.gpu


def _model(dtype, hidden=128, heads=2, layers=2, inner=256):
    torch.manual_seed(0)
    cfg = DebertaV2Config(vocab_size=500, hidden_size=hidden, num_hidden_layers=layers, num_attention_heads=heads, intermediate_size=inner,
                          max_position_embeddings=512, type_vocab_size=0, relative_attention=True, position_buckets=256,
                          max_relative_positions=512, share_att_key=True, pos_att_type=["c2p", "p2c"], norm_rel_ebd="layer_norm",
                          position_biased_input=False, layer_norm_eps=1e-7, initializer_range=0.1)
    model = FlashDebertaV2Model(cfg)
    with torch.no_grad():
        for n, p in model.named_parameters():
            if n.endswith("bias"):
                p.normal_(std=0.1)
    return model.to(device="cuda", dtype=dtype).eval()


def _ids(lens, L):
    ids = torch.randint(1, 500, (len(lens), L), generator=torch.Generator().manual_seed(L))
    for b, n in enumerate(lens):
        ids[b, n:] = 0
    return ids.cuda(), (ids != 0).long().cuda()


def _both(model, ids, mask):
    with torch.no_grad():
        fast = model._forward_native(ids, mask)
        model.encoder.pack_sequences = False
        slow = model(input_ids=ids, attention_mask=mask).last_hidden_state
        model.encoder.pack_sequences = True
        assert fast is not None
    return fast, slow


TOL = {torch.float32: 1e-5, torch.bfloat16: 2e-2, torch.float16: 3e-3}


def _check(fast, slow, mask, dtype):
    v = mask.bool()
    a, b = fast[v].double(), slow[v].double()
    assert ((a - b).norm() / b.norm()).item() <= TOL[dtype]
    assert not fast[~v].any()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("lens,L", [([1], 1), ([15], 15), ([17], 17), ([48], 48), ([64], 64), ([65], 65), ([97], 97), ([128], 128), ([129], 129),
                                    ([100, 3, 40], 100), ([256, 256], 256), ([200, 300, 13], 300)])
def test_equals_the_modules(lens, L, dtype):
    ids, mask = _ids(lens, L)
    _check(*_both(_model(dtype), ids, mask), mask, dtype)


@pytest.mark.parametrize("hidden,heads,inner", [(768, 12, 3072), (1024, 16, 4096), (64, 1, 96), (1536, 24, 128)])
@pytest.mark.parametrize("lens,L", [([40], 40), ([300, 310, 20], 310)])
def test_widths(hidden, heads, inner, lens, L):
    ids, mask = _ids(lens, L)
    _check(*_both(_model(torch.bfloat16, hidden, heads, 1, inner), ids, mask), mask, torch.bfloat16)


@pytest.mark.parametrize("hidden,heads,inner,L", [(704, 11, 3104, 50), (768, 12, 4096, 64), (768, 12, 3072, 17), (128, 2, 4128, 64)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_few_rows_with_the_normalisation_in_the_products(hidden, heads, inner, L, dtype):
    """Workgroups of one to four column blocks, the last of them short; contractions that the waves share unevenly."""
    ids, mask = _ids([L], L)
    _check(*_both(_model(dtype, hidden, heads, 2, inner), ids, mask), mask, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lens,L", [([1], 1), ([15], 15), ([17], 17), ([48], 48), ([49], 49), ([64], 64), ([20, 3, 41], 41)])
def test_few_rows_of_wider_models(lens, L, dtype):
    """Products, then residual and LayerNorm in launches of their own: one to four row tiles, and a first layer whose rows the next
    one's product reads in its own order."""
    assert _lib.load().tdb_enc_rows_fused(64, 832, 160, _lib.TDB_BF16) == 0
    ids, mask = _ids(lens, L)
    _check(*_both(_model(dtype, 832, 13, 2, 160), ids, mask), mask, dtype)


@pytest.fixture(scope="module")
def base_width():
    """Three base-sized layers: Hugging Face's model with weights as a 16-bit model holds them, in float32 and in the type."""
    def make(dtype):
        cfg = DebertaV2Config(vocab_size=500, hidden_size=768, num_hidden_layers=3, num_attention_heads=12, intermediate_size=3072,
                              max_position_embeddings=512, type_vocab_size=0, relative_attention=True, position_buckets=256,
                              max_relative_positions=512, share_att_key=True, pos_att_type=["c2p", "p2c"], norm_rel_ebd="layer_norm",
                              position_biased_input=False, layer_norm_eps=1e-7)
        torch.manual_seed(0)
        rounded = DebertaV2Model(cfg).eval()
        fill_params(rounded, seed=5)
        rounded.to(dtype)
        return rounded, copy.deepcopy(rounded).float(), patch_model(copy.deepcopy(rounded)).cuda()
    return {dtype: make(dtype) for dtype in (torch.bfloat16, torch.float16)}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lens,L", [([1], 1), ([16], 16), ([48], 48), ([20, 3, 41], 41), ([65], 65), ([200, 77, 128], 200)])
def test_as_close_to_float32_as_hugging_face(lens, L, dtype, base_width):
    """Few rows (up to 64 tokens) and tiled products: error against the float32 model no larger than that of Hugging Face's own
    run in the type, which rounds more often (measured: 0.62 to 0.73 of it)."""
    theirs, truth, ours = base_width[dtype]
    ids, mask = _ids(lens, L)
    with torch.no_grad():
        got = ours._forward_native(ids, mask).float().cpu()
        ids, mask = ids.cpu(), mask.cpu()
        ref = truth(input_ids=ids, attention_mask=mask).last_hidden_state
        hf = theirs(input_ids=ids, attention_mask=mask).last_hidden_state.float()
    v = mask.bool()
    mine, other = ((x[v] - ref[v]).norm().item() for x in (got, hf))
    print(f"{dtype} {lens}: {mine / ref[v].norm().item():.2e}, Hugging Face {other / ref[v].norm().item():.2e}")
    assert mine <= other


@pytest.mark.parametrize("dtype", [torch.int64, torch.int32, torch.bool, torch.float32, torch.bfloat16])
def test_mask_scan(dtype):
    lens = torch.randint(0, 90, (70,), generator=torch.Generator().manual_seed(1)).int()
    mask = (torch.arange(90)[None] < lens[:, None]).to(dtype).cuda()
    got, cu, ok, total, ones = _lib.host().scan_mask(mask)
    assert ok and ones and total == int(lens.sum()) and torch.equal(got.cpu(), lens)
    assert torch.equal(cu.cpu(), torch.cat([torch.zeros(1, dtype=torch.int64), lens.cumsum(0)]).int())
    holes = mask.clone()
    holes[3] = 0
    holes[3, 5] = 1
    assert not _lib.host().scan_mask(holes)[2]
    if dtype != torch.bool:
        assert not _lib.host().scan_mask(mask * 2)[4]


def test_mask_scans_of_many_threads():
    """Threads that come and go leave no pinned memory behind; threads at the same time get their own answers."""
    masks = [(torch.arange(50)[None] < torch.arange(1, 9)[:, None] + n).long().cuda() for n in range(8)]
    wrong, start = [], threading.Barrier(8)

    def scan(n, times, wait):
        if wait:
            start.wait()
        with torch.cuda.stream(torch.cuda.Stream() if wait else torch.cuda.current_stream()):
            for _ in range(times):
                lens, _, ok, total, _ = _lib.host().scan_mask(masks[n])
                if not ok or total != 36 + 8 * n or lens.tolist() != list(range(1 + n, 9 + n)):
                    wrong.append(n)

    def pinned():
        with open("/proc/self/maps") as f:
            return sum("/dev/dri/" in line or "/dev/kfd" in line for line in f)

    def run(threads):
        for t in threads:
            t.start()
        for t in threads:
            t.join()

    torch.cuda.synchronize()
    run([threading.Thread(target=scan, args=(n, 50, True)) for n in range(8)])
    before = pinned()
    for _ in range(100):
        run([threading.Thread(target=scan, args=(0, 1, False))])
    assert not wrong and pinned() - before < 20


def test_steps_aside_and_comes_back():
    model = _model(torch.bfloat16)
    ids, mask = _ids([30, 7], 30)
    dense = model.encoder.layer[1].output.dense
    with torch.no_grad():
        assert model._forward_native(ids, mask) is not None
        plan = _native_plan(model)
        assert _native_plan(model) is plan
        hook = dense.register_forward_hook(lambda m, i, o: o)
        assert _native_plan(model) is None
        hook.remove()
        assert _native_plan(model) is not None
        model.encoder.layer[0].output.dropout.train()
        assert _native_plan(model) is None
        model.eval()
        first = model._forward_native(ids, mask)
        dense.weight.mul_(1.5)
        second = model._forward_native(ids, mask)
        assert not torch.equal(first, second)
        _check(*_both(model, ids, mask), mask, torch.bfloat16)
        dense.forward = lambda x: x
        assert _native_plan(model) is None
        del dense.forward
        model.encoder.layer[1].output.dense = torch.nn.Linear(256, 128).to("cuda", torch.bfloat16).eval()
        _check(*_both(model, ids, mask), mask, torch.bfloat16)
        assert model._forward_native(ids, mask * 2) is None                    # the embeddings are scaled by such a mask
        with torch.autocast("cuda", torch.bfloat16):
            assert model._forward_native(ids, mask) is None
        with FlopCounterMode(display=False) as counter:
            model(input_ids=ids, attention_mask=mask)
        assert counter.get_total_flops() > 2 * int(mask.sum()) * 2 * (4 * 128 * 128 + 2 * 128 * 256) * 0.9
        twin = copy.deepcopy(model)
        assert torch.equal(twin._forward_native(ids, mask), model._forward_native(ids, mask))
    assert model._forward_native(ids, mask) is None                            # gradients on


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("id_type", [torch.int64, torch.int32])
@pytest.mark.parametrize("bad", [-1, 500, 2 ** 31 - 1])
def test_ids_outside_the_vocabulary(bad, id_type, dtype):
    model, (ids, mask) = _model(dtype), _ids([30, 7, 12], 30)
    ids = ids.to(id_type)
    run = lambda mask: model._forward_native(ids, mask)                          # (the modules never see such ids)
    with torch.no_grad():
        good = run(mask)
        ids[1, 7], ids[2, 29] = bad, bad                                        # padding
        assert torch.equal(run(mask.clone()), good)
        ids[1, 6] = bad
        with pytest.raises(IndexError, match="500"):
            run(mask.clone())
        out = run(mask)                                                         # measured before: nothing is read back
        assert out[1, :7].isnan().all() and torch.equal(out[0], good[0]) and torch.equal(out[2], good[2])
        ids[1, 7] = ids[2, 29] = 5
        out = run(None)
        assert out[1].isnan().all() and not out[0].isnan().any() and not out[2].isnan().any()


@pytest.mark.parametrize("kind", ["full", "declared", "measured"])
def test_nothing_computed_under_capture_is_kept(kind):
    """A forward captured before any eager one: the eager ones after it do not find what only a replay computes."""
    model, warm = _model(torch.bfloat16), _model(torch.bfloat16)
    ids, mask = _ids([30, 30, 30] if kind == "full" else [30, 7, 12], 30)
    declared = None
    if kind == "declared":
        declared = declare_right_padded(mask.clone(), mask.sum(-1, dtype=torch.int32), int(mask.sum()))
    elif kind == "measured":
        declared = mask.clone()
    with torch.no_grad():
        want = warm._forward_native(ids, mask)                     # (kernels and position tables are there from here on)
        if kind == "measured":
            warm._forward_native(ids, declared)
        graph = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph):
            out = model._forward_native(ids, declared)
        assert out is not None
        junk = torch.full((1 << 24,), float("nan"), device="cuda")
        assert torch.equal(model._forward_native(ids, declared), want)
        for _ in range(3):
            out.zero_()
            graph.replay()
            assert torch.equal(out, want) and torch.equal(model._forward_native(ids, declared), want)
        del junk


def test_a_plan_serves_other_streams():
    model, twin = _model(torch.bfloat16), _model(torch.bfloat16)
    ids, mask = _ids([30, 7, 12], 30)
    side = torch.cuda.Stream()
    with torch.no_grad():
        want = twin._forward_native(ids, None)
        torch.cuda.synchronize()
        torch.cuda._sleep(20_000_000)                              # the first call's weights are concatenated behind this
        first = model._forward_native(ids, None)
        with torch.cuda.stream(side):
            second = model._forward_native(ids, None)
        torch.cuda.synchronize()
    assert torch.equal(first, want) and torch.equal(second, want)


@pytest.mark.parametrize("lengths,total", [([30, 7, 12], 60), ([30, 7, 12], 20), ([60, -9, 70], 80)])
def test_declared_lengths_that_do_not_fit(lengths, total):
    """Nobody verifies them and the results mean nothing; every access stays inside."""
    model, (ids, mask) = _model(torch.bfloat16), _ids([30, 7, 12], 30)
    with torch.no_grad():
        want = model._forward_native(ids, mask)
        wrong = declare_right_padded(mask.clone(), torch.tensor(lengths, dtype=torch.int32, device="cuda"), total)
        assert model._forward_native(ids, wrong).shape == want.shape
        assert torch.equal(model._forward_native(ids, mask.clone()), want)


def test_refused_heads_raise_the_operators_error():
    model, (ids, mask) = _model(torch.bfloat16, hidden=72, heads=6, inner=96), _ids([30, 7, 12], 30)
    for m in (mask, torch.ones_like(mask)):
        with torch.no_grad(), pytest.raises(ValueError, match="head_dim 12"):
            model(input_ids=ids, attention_mask=m)


def test_boundaries_it_does_not_take():
    model, (ids, mask) = _model(torch.bfloat16), _ids([30, 7, 12], 30)
    with torch.no_grad():
        model._forward_native(ids, mask)
        plan, cu = _native_plan(model), torch.tensor([0, 30, 37, 49], dtype=torch.int32, device="cuda")
        encode = _lib.host().encode
        assert encode(plan, ids, cu, 49) is not None
        for bad in (cu.long(), cu.cpu(), cu[:3], cu[None], cu.repeat_interleave(2)[::2], [0, 30, 37, 49]):
            assert encode(plan, ids, bad, 49) is None


class _LastHidden(torch.nn.Module):
    def __init__(self, model):
        super().__init__()
        self.model = model

    def forward(self, ids, mask):
        return self.model(input_ids=ids, attention_mask=mask).last_hidden_state


@pytest.mark.parametrize("lens", [[30, 7, 12], [30, 30, 30]])
def test_traced_model_replays_on_other_inputs(lens):
    model = _model(torch.float32)
    run = _LastHidden(model).eval()
    with torch.no_grad():
        example = _ids(lens, 30)
        run(*example)
        traced = torch.jit.trace(run, example, check_trace=False)
        for other in ([30, 7, 12], [3, 30, 29], [1, 1, 1]):
            ids, mask = _ids(other, 30)
            ids = torch.where(ids > 0, 500 - ids, 0)
            got, v = traced(ids, mask), mask.bool()
            torch.testing.assert_close(got[v], _both(model, ids, mask)[1][v], rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("dtype,code", [(torch.bfloat16, 1), (torch.float16, 2)])
@pytest.mark.parametrize("tile", range(7))
def test_product_tiles(tile, dtype, code):
    """Every tile of the products (0: the one the kernel chooses) where it ends inside the output, and with fewer steps of the
    contraction than it has stages, whole and in parts."""
    lib, ptr = _lib.load(), lambda t: C.c_void_p(t.data_ptr())
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    for M, N, K in [(1, 8, 64), (33, 72, 128), (127, 136, 192), (130, 264, 448), (513, 520, 832)]:
        g = torch.Generator(device="cuda").manual_seed(M)
        x = torch.randn(M, K, device="cuda", generator=g).to(dtype)
        w, b = (torch.randn(N, K, device="cuda", generator=g) / K ** 0.5).to(dtype), torch.randn(N, device="cuda", generator=g).to(dtype)
        y, parts = torch.full((M, N), 7., device="cuda", dtype=dtype), torch.full((2, M, N), 7., device="cuda")
        ref = x.double() @ w.double().t()
        run = lambda flags, splits, out: lib.tdb_enc_gemm(ptr(x), ptr(w), ptr(b), flags | tile << 8, splits, M, N, K, code, ptr(out), stream)
        eps = torch.finfo(dtype).eps
        assert run(0, 1, y) == 0
        torch.testing.assert_close(y.double(), ref + b.double(), rtol=eps, atol=eps)
        assert run(4, 1, y) == 0
        torch.testing.assert_close(y.double(), torch.nn.functional.gelu(ref + b.double()), rtol=eps, atol=eps)
        if K > 64:
            assert run(0, 2, parts) == 0
            torch.testing.assert_close(parts.double().sum(0), ref, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("dtype,code", [(torch.bfloat16, 1), (torch.float16, 2)])
@pytest.mark.parametrize("tile,M,N", [(5, 4229, 2056), (5, 257 * 128, 256), (5, 8192, 3080), (6, 4229, 4104), (7, 577, 392), (7, 7000, 1032)])
@pytest.mark.parametrize("K", [192, 256, 320, 448])
def test_tile_after_tile(tile, M, N, K, dtype, code):
    """More large tiles than compute units: one more, some workgroups with one more than others, ends inside the output; steps of the
    contraction one to four more than stages, and as many (which one workgroup a tile takes); and the tile of 192 rows."""
    lib, ptr = _lib.load(), lambda t: C.c_void_p(t.data_ptr())
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    g = torch.Generator(device="cuda").manual_seed(K)
    x = torch.randn(M, K, device="cuda", generator=g).to(dtype)
    w, b = (torch.randn(N, K, device="cuda", generator=g) / K ** 0.5).to(dtype), torch.randn(N, device="cuda", generator=g).to(dtype)
    ref, eps = x.double() @ w.double().t() + b.double(), torch.finfo(dtype).eps
    for flags in (0, 4):
        y = torch.full((M, N), 7., device="cuda", dtype=dtype)
        assert lib.tdb_enc_gemm(ptr(x), ptr(w), ptr(b), flags | tile << 8, 1, M, N, K, code, ptr(y), stream) == 0
        torch.testing.assert_close(y.double(), torch.nn.functional.gelu(ref) if flags else ref, rtol=eps, atol=eps)


@pytest.mark.parametrize("dtype,code", [(torch.bfloat16, 1), (torch.float16, 2)])
def test_gelu_over_its_range(dtype, code):
    """GELU of the products' epilogue, through a product with a unit vector: half a unit in the last place of the result, the
    fit's 6e-6 and, below -5, its 3e-10."""
    lib, ptr = _lib.load(), lambda t: C.c_void_p(t.data_ptr())
    v = torch.cat([torch.linspace(-9, 9, 20001), torch.tensor([0., -20., 20., -6e4, 6e4, float("inf"), -float("inf"), float("nan")])]).to(dtype).cuda()
    x, w, b = torch.zeros(len(v), 64, dtype=dtype, device="cuda"), torch.zeros(8, 64, dtype=dtype, device="cuda"), torch.zeros(8, dtype=dtype, device="cuda")
    x[:, 0], w[:, 0] = v, 1
    y = torch.empty(len(v), 8, dtype=dtype, device="cuda")
    assert lib.tdb_enc_gemm(ptr(x), ptr(w), ptr(b), 4, 1, len(v), 8, 64, code, ptr(y), C.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    ref = torch.nn.functional.gelu(v.double())[:, None].expand(-1, 8)
    smallest = 2.0 ** -24 if dtype == torch.float16 else 0.0
    torch.testing.assert_close(y.double(), ref, rtol=torch.finfo(dtype).eps / 2 + 6e-6, atol=smallest / 2 + 3e-10, equal_nan=True)


def test_product_limits():
    lib = _lib.load()
    for M, N, K, dtype in [(16, 8, 96, 1), (16, 12, 64, 1), (0, 8, 64, 1), (16, 8, 64, 0), (1 << 16, 8, 1 << 15, 1)]:
        assert lib.tdb_enc_gemm_splits(M, N, K, dtype) == 0
        assert lib.tdb_enc_gemm(None, None, None, 0, 1, M, N, K, dtype, None, None) != 0
    assert lib.tdb_enc_gemm(None, None, None, 0, 2, 16, 8, 64, 1, None, None) != 0       # more parts than steps
