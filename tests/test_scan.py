"""The native reader of tensor lists: what it takes, what it leaves to the callers' own loops, and that both give the same step."""
import numpy as np
import pytest
import torch

from lmms_engine_amd import _abi
from tests.test_gpu_parity import env  # noqa: F401


def test_cpu_tensors_and_other_things_are_left_to_the_caller():
    scan = _abi.scan()
    p = torch.nn.Parameter(torch.zeros(3, 4))
    p.grad = torch.ones(3, 4)
    state = {p: {"momentum_buffer": torch.zeros(3, 4), "exp_avg": torch.zeros(3, 4), "exp_avg_sq": torch.zeros(3, 4), "step": 4}}
    for params in ([p], (p,), [], [None], "p", [torch.nn.Parameter(torch.zeros(0))]):
        assert scan.grads(params, 16384) is None
        assert scan.muon(params, state) is None or params == []
        assert scan.adam(params, state, 16384) is None
    assert scan.muon([p], None) is None and scan.adam([p], [], 16384) is None and scan.grads([p], 0) is None
    assert state[p]["step"] == 4


def test_a_module_for_another_torch_is_refused(monkeypatch):
    scan = _abi.scan()
    assert scan.torch_version == torch.__version__
    monkeypatch.setattr(_abi, "_scan", None)
    monkeypatch.setattr(torch, "__version__", "0.0")
    with pytest.raises(_abi.MuonHipError, match="built for torch"):
        _abi.scan()


def test_nothing_counts_as_built_while_a_library_is_missing(monkeypatch):
    from lmms_engine_amd import build

    assert build.built()
    for name in ("LIB", "SCAN_LIB"):
        with monkeypatch.context() as m:
            m.setattr(build, name, "/nonexistent/" + name)
            assert not build.built()


@pytest.mark.parametrize("where", ["subclass", "class", "instance"])
@pytest.mark.parametrize("name", ["_get_work_class", "_init_muon_state"])
def test_methods_of_the_callers_own_are_asked(monkeypatch, where, name):
    """A step reads its lists in native code only where nobody has replaced the methods that choose a parameter's work and make its state."""
    from lmms_engine_amd import muon_utils

    started = []

    class OwnWork:
        def __init__(self, param, state, group, index):
            self.param = param

        def start(self):
            started.append(self.param)

        def finish(self):
            pass

    def own(*args):  # (self is the first argument but for an instance's)
        if name == "_get_work_class":
            return OwnWork, 1
        started.append(args[-1])
        raise KeyboardInterrupt

    monkeypatch.setattr(_abi, "scan", lambda: pytest.fail("read in native code"))
    cls = type("Sub", (muon_utils.Muon,), {name: own}) if where == "subclass" else muon_utils.Muon
    p = torch.nn.Parameter(torch.zeros(3, 4))
    p.grad = torch.ones(3, 4)
    opt = cls([dict(params=[p], use_muon=True)])
    assert (where == "subclass") != opt._plain_work()
    if where == "class":
        monkeypatch.setattr(muon_utils.Muon, name, own)
    elif where == "instance":
        monkeypatch.setattr(opt, name, own)
    if name == "_get_work_class":
        opt.step()
    else:
        with pytest.raises(KeyboardInterrupt):
            opt.step()
    assert len(started) == 1 and started[0] is p


def _set(dev, dtype, seed=0):
    g = torch.Generator().manual_seed(seed)
    shapes = [(96, 40), (128, 256), (96, 40), (300, 20), (128, 256)]
    mats = [torch.nn.Parameter((0.02 * torch.randn(*s, generator=g)).to(dtype).to(dev)) for s in shapes]
    rest = [torch.nn.Parameter(torch.randn(n, generator=g).to(dtype).to(dev)) for n in (5, 16384 * 2 + 3, 7)]
    for p in mats + rest:
        p.grad = torch.randn(p.shape, generator=g).to(dtype).to(dev)
    return mats, rest


def _optimizer(mu, mats, rest, mdtype=None):
    return mu.Muon([dict(params=list(mats), use_muon=True, lr=0.02, momentum=0.95, nesterov=True, weight_decay=0.01, ns_steps=5, rms_scale=True),
                    dict(params=list(rest), use_muon=False, lr=1e-3, betas=(0.9, 0.95), eps=1e-8, weight_decay=0.01)], momentum_dtype=mdtype)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,mdtype", [(torch.float32, None), (torch.bfloat16, torch.float32)])
def test_step_and_clipping_equal_the_callers_own_loops(env, monkeypatch, dtype, mdtype):
    from lmms_engine_amd.clip_grad import clip_grad_norm_

    mu, dev = env["mu"], env["dev"]

    class Loops:
        grads = muon = adam = staticmethod(lambda *a: None)

    out = []
    for own in (False, True):
        mats, rest = _set(dev, dtype)
        opt = _optimizer(mu, mats, rest, mdtype)
        opt.step()  # makes the state: nobody's fast path
        scan = _abi.scan()
        assert scan.muon(opt.param_groups[0]["params"], opt.state) and scan.grads(mats + rest, 16384)
        with monkeypatch.context() as m:
            if own:
                m.setattr(_abi, "scan", lambda: Loops)
            totals = []
            for _ in range(3):
                totals.append(clip_grad_norm_(mats + rest, 1.0).clone())
                opt.step()
        torch.cuda.synchronize()
        out.append((mats + rest, totals, [opt.state[p]["step"] for p in rest], [opt.state[p]["momentum_buffer"] for p in mats],
                    [p.grad for p in mats + rest], [opt.state[p]["exp_avg_sq"] for p in rest]))
    a, b = out
    assert a[2] == b[2] == [4, 4, 4]
    for x, y in zip(a[0] + a[1] + a[3] + a[4] + a[5], b[0] + b[1] + b[3] + b[4] + b[5]):
        assert torch.equal(x.detach(), y.detach())


@pytest.mark.gpu
@pytest.mark.parametrize("first", [torch.float32, torch.bfloat16])
def test_clipping_gradients_of_two_dtypes_and_of_none_equals_the_callers_own_loop(env, monkeypatch, first):
    from lmms_engine_amd.clip_grad import clip_grad_norm_

    class Loops:
        grads = staticmethod(lambda *a: None)

    dev, out = env["dev"], []
    other = torch.bfloat16 if first == torch.float32 else torch.float32
    for own in (False, True):
        g = torch.Generator().manual_seed(5)
        ps = []
        for n, dtype in ((7, first), (16384 + 5, other), (300, first), (16384 * 3, first), (64, other), (9, other)):
            p = torch.nn.Parameter(torch.zeros(n, dtype=dtype, device=dev))
            p.grad = torch.randn(n, generator=g).to(dtype).to(dev)
            ps.append(p)
        ps[2].grad = ps[5].grad = None
        ps.insert(0, torch.nn.Parameter(torch.zeros(4)))  # no gradient, not on the device either
        lists = _abi.scan().grads(ps, 16384)[1]
        assert [(code, n, chunks) for code, n, chunks, _ in lists] == [(_abi.dtype_code(first), 2, 4), (_abi.dtype_code(other), 2, 3)]
        with monkeypatch.context() as m:
            if own:
                m.setattr(_abi, "scan", lambda: Loops)
            totals = [clip_grad_norm_(ps, 1.0, norm_type=t) for t in (2.0, float("inf"))]
        torch.cuda.synchronize()
        out.append((totals, [p.grad for p in ps]))
    for x, y in zip(out[0][0] + out[0][1], out[1][0] + out[1][1]):
        assert (x is None) == (y is None) and (x is None or (x.dtype == y.dtype and torch.equal(x, y)))
    assert out[0][0][0].dtype == torch.float32


@pytest.mark.gpu
def test_addresses_sizes_and_order(env):
    mats, rest = _set(env["dev"], torch.float32)
    opt = _optimizer(env["mu"], mats, rest)
    opt.step()
    ps = opt.param_groups[0]["params"]
    for dev, rows, cols, pc, gc, mc, n, p, g, m in _abi.scan().muon(ps, opt.state):
        mine = [q for q in ps if tuple(q.shape) == (rows, cols)]
        assert (dev, pc, gc, mc, n) == (mats[0].get_device(), 0, 0, 0, len(mine))
        for words, ts in ((p, mine), (g, [q.grad for q in mine]), (m, [opt.state[q]["momentum_buffer"] for q in mine])):
            assert np.frombuffer(words, np.int64).tolist() == [t.data_ptr() for t in ts]
    _, ((code, n, chunks, words),) = _abi.scan().grads(rest, 16384)
    assert (code, n, chunks) == (0, 3, 1 + 3 + 1)
    assert np.frombuffer(words, np.int64).tolist() == [p.grad.data_ptr() for p in rest] + [p.numel() for p in rest] + [0, 1, 4, 5]


@pytest.mark.gpu
def test_lists_that_need_a_decision_are_left_to_the_caller(env):
    dev, scan = env["dev"], _abi.scan()
    for change in ("no grad", "strided grad", "strided parameter", "grad of another dtype", "no state", "shape", "subclass", "float step", "twice"):
        mats, rest = _set(dev, torch.float32)
        opt = _optimizer(env["mu"], mats, rest)
        opt.step()
        p, q, params = mats[0], rest[1], list(rest)
        if change == "no grad":
            p.grad = q.grad = None
        elif change == "strided grad":
            p.grad = torch.randn(40, 96, device=dev).t()
            q.grad = torch.randn(q.numel(), 2, device=dev)[:, 0]
        elif change == "strided parameter":
            p.data = torch.randn(40, 96, device=dev).t()
            q.data = torch.randn(q.numel(), 2, device=dev)[:, 0]
        elif change == "grad of another dtype":
            p.data, q.data = p.data.bfloat16(), q.data.bfloat16()
            opt.state[p]["momentum_buffer"] = opt.state[p]["momentum_buffer"].half()
        elif change == "no state":
            opt.state[p], opt.state[q] = {}, {}
        elif change == "shape":
            opt.state[p]["momentum_buffer"] = torch.zeros(40, 96, device=dev)
            opt.state[q]["exp_avg"] = torch.zeros(3, device=dev)
        elif change == "subclass":
            class Sub(torch.nn.Parameter):
                pass
            for old in (p, q):
                new = Sub(old.detach().clone())
                new.grad, opt.state[new] = old.grad, opt.state[old]
                mats, params = [new if t is old else t for t in mats], [new if t is old else t for t in params]
        elif change == "float step":
            opt.state[q]["step"] = 2.0
            opt.state[p]["momentum_buffer"] = None
        elif change == "twice":
            params.append(q)
            opt.state[p]["momentum_buffer"] = opt.state[p]["momentum_buffer"].cpu()
        before = [opt.state[t].get("step") for t in rest]
        held = []
        if change in ("strided grad", "subclass"):
            assert scan.grads(mats, 16384, held) is None and scan.grads(params, 16384, held) is None and not held, change
        assert scan.muon(mats, opt.state, held) is None, change
        assert scan.adam(params, opt.state, 16384, held) is None and not held, change
        assert [opt.state[t].get("step") for t in rest] == before, change


@pytest.mark.gpu
def test_memory_lives_until_the_last_launch(env, monkeypatch):
    """Gradients that their parameters give up between the reading of the addresses and the launches (another thread may, while a call
    waits or launches) stay allocated until the call is through."""
    from lmms_engine_amd.clip_grad import clip_grad_norm_

    mu, dev = env["mu"], env["dev"]
    mats = [torch.nn.Parameter(torch.zeros(256, 4096, device=dev)) for _ in range(4)]
    rest = [torch.nn.Parameter(torch.zeros(1 << 20, device=dev)) for _ in range(4)]
    both = _optimizer(mu, mats, rest)
    stream_ptr, seen = _abi.stream_ptr, []

    def drop(device):
        before = torch.cuda.memory_allocated()
        for p in dropped:
            p.grad = None
        seen.append(before - torch.cuda.memory_allocated())
        return stream_ptr(device)

    def set_grads():
        for p in mats + rest:
            p.grad = torch.ones_like(p)

    set_grads()
    both.step()  # makes the state
    for call, dropped in ((lambda: clip_grad_norm_(mats + rest, 1.0, error_if_nonfinite=True), mats + rest), (both.step, mats),
                          (lambda: both._adam_group_step(both.param_groups[1]), rest)):
        set_grads()
        del seen[:]
        with monkeypatch.context() as m:
            m.setattr(_abi, "stream_ptr", drop)
            call()
        assert seen and not any(seen), seen
        assert all(p.grad is None for p in dropped)
    torch.cuda.synchronize()
