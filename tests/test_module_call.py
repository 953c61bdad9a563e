"""QuantLinear's C call (csrc/python_call.cpp): what it takes by itself and what it hands to nn.Module.__call__ give the
same numbers, and the module's ways of being changed or watched still reach it."""
import pytest
import torch

from autogptq.tvm_amd import _lib, ops
from autogptq.tvm_amd.qlinear import QuantLinear
from tests.parity_util import assert_tight, expected_output, expected_weight, layer

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


@pytest.mark.parametrize("bits,desc_act,M", [(4, False, 1), (3, True, 4), (8, True, 9), (4, True, 40)])
def test_the_call_in_c_equals_forward(dev, bits, desc_act, M):
    L = layer(4100 + M, 512, 96, bits, 128, desc_act, M=M, bias=True)
    q = QuantLinear(bits, 128, 512, 96, True)
    q.load_state_dict({k: L[k] for k in ("qweight", "qzeros", "scales", "g_idx", "bias")})
    q = q.to(dev)
    x = L["x"].to(dev)
    first = q(x)                                   # no route yet: through nn.Module.__call__
    assert isinstance(q._routes[M][3], ops.CALL.BoundCall)
    assert_tight(first, expected_output(L), "first call")
    shapes = [(M, 512), (1, M, 512), (M, 1, 512), (1, 1, M, 512)] + ([(512,)] if M == 1 else [])
    for shape in shapes:
        y = q(x.view(shape))
        assert y.shape == shape[:-1] + (96,) and y.dtype == torch.float16 and not y.requires_grad
        assert torch.equal(y.view(M, 96), first)
    # what it does not take: another dtype, a strided x, a keyword, a gradient
    assert torch.equal(q(x.float()), first)
    wide = torch.empty((M, 1024), dtype=torch.float16, device=dev)
    wide[:, ::2] = x
    assert torch.equal(q(wide[:, ::2]), first) and torch.equal(q(x=x), first)
    assert q(x.clone().requires_grad_(True)).requires_grad
    with torch.no_grad():
        assert torch.equal(q(x.clone().requires_grad_(True)), first)
    with pytest.raises(Exception):
        q(x[:, :256].contiguous())
    with pytest.raises(RuntimeError, match="no CPU fallback"):
        q(x.cpu())


def test_hooks_replaced_buffers_and_instance_forward_are_seen(dev):
    L = layer(4150, 512, 96, 4, 128, True, M=2, bias=False)
    q = QuantLinear(4, 128, 512, 96, False)
    q.load_state_dict({k: L[k] for k in ("qweight", "qzeros", "scales", "g_idx")})
    q = q.to(dev)
    x = L["x"].to(dev)
    first = q(x)
    assert torch.equal(q(x), first)
    seen = []
    for register in (q.register_forward_hook, torch.nn.modules.module.register_module_forward_hook):
        h = register(lambda m, i, o: seen.append(m))
        q(x)
        h.remove()
        q(x)
    h = q.register_forward_pre_hook(lambda m, i: seen.append(m))
    q(x)
    h.remove()
    assert seen == [q, q, q]
    q.forward = lambda t: "replaced"
    assert q(x) == "replaced"
    del q.forward

    class Sub(QuantLinear):
        def forward(self, t):
            return "subclass"

    s = Sub(4, 128, 512, 96, False).to(dev)
    s._routes = dict(q._routes)
    assert s(x) == "subclass"
    q.scales.mul_(2)                               # written in place: the copies are made again
    assert torch.allclose(q(x).float(), 2 * first.float(), rtol=1e-3, atol=1e-3)
    q._buffers["scales"] = q.scales * 0            # swapped behind the module's back
    assert float(q(x).abs().max()) == 0.0


def module_of(L, dev, **kw):
    q = QuantLinear(L["bits"], L["group_size"], L["K"], L["N"], L.get("bias") is not None, **kw)
    q.load_state_dict({k: L[k] for k in ("qweight", "qzeros", "scales", "g_idx", "bias") if L.get(k) is not None})
    return q.to(dev)


@pytest.mark.parametrize("way", ["operator", "front end", "gradient", "module"])
def test_threads_on_one_stream_do_not_mix_their_launches(dev, way):
    """A call of a pack pass, a product and a sum hands them x and partial sums through its stream's workspace: the launches
    of another thread's call do not come between."""
    import threading

    M, K, N = 40, 2048, 1056
    L = layer(4250, K, N, 4, 128, True, M=M)
    q = module_of(L, dev)
    qtile, sz, xsrc, kinv = q.prepare_tiled()
    plan = _lib.select_tiled(M, K, N, 4, 128)
    assert plan.workspace_bytes and q.prepare_transposed() is not None
    call = {"operator": lambda t: torch.ops.gptq_hip.gemm_tiled(t, qtile, sz, xsrc, kinv, None, 4, 128),
            "front end": lambda t: ops.gemm_tiled(t, qtile, sz, xsrc, kinv, None, 4, 128, plan=plan),
            "gradient": q.grad_input, "module": q}[way]
    width = N if way == "gradient" else K
    xs = [torch.randn(M, width, dtype=torch.float16, device=dev) for _ in range(4)]
    want = [call(x) for x in xs]
    torch.cuda.synchronize()
    wrong = [0] * len(xs)

    def work(i):
        got = [call(xs[i]) for _ in range(200)]        # (every thread on the same, the default, stream)
        wrong[i] = sum(not torch.equal(y, want[i]) for y in got)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(xs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert wrong == [0] * len(xs)


def test_other_threads_run_while_a_call_allocates_and_launches(dev):
    """The call gives the interpreter free around its allocation and launch.  The switch interval is far beyond the test, so
    that another thread advances only where the call itself lets it; the emptied cache makes the allocation a long one."""
    import sys
    import threading
    import time

    L = layer(4200, 512, 16384, 4, 128, False, M=64)
    q, x = module_of(L, dev), L["x"].to(dev)
    for _ in range(3):
        y = q(x)
    beat, stop = [0], threading.Event()

    def run():
        while not stop.is_set():
            beat[0] += 1
            time.sleep(0)

    interval = sys.getswitchinterval()
    sys.setswitchinterval(60.0)
    advanced = 0
    t = threading.Thread(target=run)
    t.start()
    try:
        for _ in range(50):
            y = None
            torch.cuda.empty_cache()
            before = beat[0]
            y = q(x)
            advanced += beat[0] != before
    finally:
        stop.set()
        sys.setswitchinterval(interval)
        t.join()
    assert advanced > 0 and y is not None


@pytest.mark.parametrize("M", [1, 8, 40, 1300])
def test_rows_at_an_odd_offset_are_taken(dev, M):
    """A contiguous view of a larger tensor need not be aligned for the kernels' 16-byte loads: on every route, and as a
    gradient."""
    K, N = 2048, 4128
    L = layer(9710, K, N, 4, 128, True, M=M, bias=True)
    q, x = module_of(L, dev), L["x"].to(dev)
    want = q(x)
    gy = torch.randn(M, N, generator=torch.Generator().manual_seed(3)).half().to(dev)
    want_t = q.grad_input(gy)
    for offset in (1, 4):
        odd = torch.empty(M * K + 8, dtype=torch.float16, device=dev)[offset:offset + M * K].view(M, K).copy_(x)
        assert odd.data_ptr() % 16 and odd.is_contiguous()
        assert torch.equal(q(odd), want) and torch.equal(q(odd.view(M, 1, K)).view(M, N), want)
        if q.route(M) == "tiled":
            qtile, sz, xsrc, kinv = q.prepare_tiled()
            assert torch.equal(torch.ops.gptq_hip.gemm_tiled(odd, qtile, sz, xsrc, kinv, q.bias, 4, 128), want)
        odd_t = torch.empty(M * N + 8, dtype=torch.float16, device=dev)[offset:offset + M * N].view(M, N).copy_(gy)
        assert torch.equal(q.grad_input(odd_t), want_t)
        xg = odd.clone().requires_grad_(True)
        q(xg).backward(odd_t)
        assert torch.equal(xg.grad, want_t)


def python_frames(fn):
    """The names of the Python functions that a call of ``fn`` enters."""
    import sys

    names = []
    sys.setprofile(lambda frame, event, arg: event == "call" and names.append(frame.f_code.co_name))
    try:
        fn()
    finally:
        sys.setprofile(None)
    return names


def test_methods_replaced_on_the_classes_are_seen(dev, monkeypatch):
    L = layer(4160, 512, 96, 4, 128, True, M=2)
    q, x = module_of(L, dev), L["x"].to(dev)
    first = q(x)
    call = lambda: q(x)
    for owner, name in ((QuantLinear, "forward"), (QuantLinear, "__call__"), (QuantLinear, "_call_impl"),
                        (torch.nn.Module, "__call__"), (torch.nn.Module, "_call_impl")):
        original, seen = getattr(owner, name), []
        with monkeypatch.context() as m:
            m.setattr(owner, name, lambda self, *a: (seen.append(name), original(self, *a))[1])
            assert torch.equal(q(x), first) and seen == [name]
        assert torch.equal(q(x), first) and seen == [name]
        assert python_frames(call) == ["<lambda>"]            # untouched again: the call in C
    q._call_impl = lambda *a: "instance"
    assert q(x) == "instance"


@pytest.mark.parametrize("M,desc_act", [(1, True), (9, True), (600, True), (600, False)])
def test_the_first_call_of_a_layer_waits_for_the_gpu_once(dev, M, desc_act):
    import warnings

    L = layer(9730 + M, 2048, 4128, 4, 128, desc_act, M=M, bias=True)
    q, x = module_of(L, dev), L["x"].to(dev).requires_grad_(True)
    gy = torch.randn(M, 4128, device=dev, dtype=torch.float16)
    torch.cuda.synchronize()
    with warnings.catch_warnings(record=True) as seen:
        warnings.simplefilter("always")
        torch.cuda.set_sync_debug_mode("warn")
        try:
            y = q(x)
            gx, = torch.autograd.grad(y, x, gy)
        finally:
            torch.cuda.set_sync_debug_mode("default")
    assert sum("called a synchronizing" in str(w.message) for w in seen) == 1
    assert_tight(y.detach(), expected_output(L), "first call")
    assert_tight(gx, gy.float().cpu() @ expected_weight(L).float().t(), "first gradient")


@pytest.mark.parametrize("bits,K,M,desc_act,path", [(4, 1024, 4, True, "tiled"), (3, 4224, 12, True, "sorted"), (4, 1024, 12, False, "plain")])
@pytest.mark.parametrize("known", [False, True])
def test_what_records_a_call_sees_the_operator(dev, bits, K, M, desc_act, path, known):
    """torch.jit.trace, dispatch modes, make_fx and fake tensors get the operator of the route, whether the layer knows the row
    count already or has its copies to prepare: not a constant, and no allocation without what fills it."""
    import warnings

    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.fx.experimental.proxy_tensor import make_fx
    from torch.utils._python_dispatch import TorchDispatchMode

    N = 416
    L = layer(4300 + M, K, N, bits, 128, desc_act, M=M, bias=True)
    x = L["x"].to(dev)
    other = torch.randn_like(x)
    one = module_of(L, dev)
    first, want = one(x), one(other)

    def module():
        q = module_of(L, dev).eval()
        if known:
            assert q.route(M) == path and torch.equal(q(x), first) and torch.equal(q(x), first)
        return q

    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        traced = torch.jit.trace(module(), x, check_trace=False)
    assert torch.equal(traced(other), want) and torch.equal(traced(x), first)

    class Seen(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            names.append(str(func))
            return func(*args, **(kwargs or {}))

    names, q = [], module()
    with Seen():
        assert torch.equal(q(x), first)
    assert [n for n in names if n.startswith("gptq_hip.gemm")]
    graph = make_fx(module())(x)
    assert torch.equal(graph(other), want) and any(str(n.target).startswith("gptq_hip.gemm") for n in graph.graph.nodes)
    q = module()
    with FakeTensorMode(allow_non_fake_inputs=True) as fake:
        assert q(fake.from_tensor(x)).shape == (M, N)
    assert torch.equal(q(x), first)
    with pytest.raises(RuntimeError):                       # (no rule for it, and never was one)
        torch.func.vmap(module())(torch.stack((x, other)))


@pytest.mark.parametrize("known", [False, True])
def test_compiled_models_run_the_layer_between_their_graphs(dev, known):
    import warnings

    L = layer(4350, 512, 96, 4, 128, True, M=4, bias=True)
    q, x = module_of(L, dev).eval(), L["x"].to(dev)
    net = torch.nn.Sequential(q, torch.nn.ReLU())
    want = torch.relu(module_of(L, dev)(x))
    if known:
        assert torch.equal(net(x), want)
    with warnings.catch_warnings(), torch.no_grad():
        warnings.simplefilter("ignore")
        compiled = torch.compile(net, backend="eager")
        assert torch.equal(compiled(x), want) and torch.equal(compiled(2 * x), net(2 * x))
    torch._dynamo.reset()
