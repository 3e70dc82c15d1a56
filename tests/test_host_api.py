"""Host-side logic without a GPU: the C ABI exports what include/pam_hip.h declares, and the
autograd layer (same formulas as the reference's pam/cuda_bindings.py) composes kernel calls
correctly.  The kernels are replaced by a stand-in built on the CPU oracle, so only the
plumbing is under test here; the kernels themselves are checked on the GPU."""
import ctypes
import math
import pathlib
import re

import numpy as np
import pytest
import torch

import pam_amd
from pam_amd import _abi, cuda_bindings, pam_ops
from _util import assert_same_bits

ROOT = pathlib.Path(__file__).resolve().parent.parent


def test_library_exports_every_declared_symbol():
    header = (ROOT / "include" / "pam_hip.h").read_text()
    declared = set(re.findall(r"\b(pam_hip_[a-z0-9_]+)\s*\(", header))
    assert len(declared) == 42
    # measurement probes and the tuning hook live in a header of their own, not in the drop-in interface
    probes = set(re.findall(r"\b(pam_hip_[a-z0-9_]+)\s*\(", (ROOT / "include" / "pam_hip_probe.h").read_text()))
    assert probes == {"pam_hip_issue_probe", "pam_hip_issue_probe_lds", "pam_hip_set_tuning"} and not (probes & declared)
    declared |= probes
    lib = ctypes.CDLL(str(_abi.library_path()))
    missing = [name for name in sorted(declared) if not hasattr(lib, name)]
    assert not missing, f"declared in pam_hip.h but not exported: {missing}"
    # the fourteen entry points of the reference's extension module, one to one (pam/cuda_kernels.cu:932-947)
    for name in ("pam_fwd pam_bwd pad_fwd pad_bwd pam_matmul_fwd pam_bmm_fwd pam_matmul_bwd pam_bmm_bwd "
                 "standard_matmul standard_bmm pa_exp_fwd pa_exp_bwd pa_log_fwd pa_log_bwd").split():
        assert "pam_hip_" + name in declared and hasattr(_abi.HipKernels, name)
    assert set(_abi.exported_symbols()) <= declared
    assert _abi.load_library().pam_hip_abi_version() == 2
    # the library under test was built from the sources of this tree
    from pam_amd import build as builder
    assert _abi.load_library().pam_hip_source_hash().decode() == builder.source_hash()


def test_log2_of_the_usual_bases_is_pinned():
    """pa_exp / pa_log scale by the fp32 constant log2(base); one unit of the last place in it moves every result.
    The goldens of tests/golden/exp_log.npz were written with torch.log2(torch.tensor(base)) on the CPU: the
    library's constant, the oracle's and torch's must be these bit patterns."""
    import numpy as np
    import torch
    from oracle import pam_oracle
    lib = _abi.load_library()
    for base, want in ((math.e, 0x3fb8aa3b), (10.0, 0x40549a78), (0.5, 0xbf800000), (2.0, 0x3f800000), (3.0, 0x3fcae00d)):
        for got in (lib.pam_hip_log2_base(base), pam_oracle.log2_base(base), torch.log2(torch.tensor(base, dtype=torch.float32)).item()):
            assert np.float32(got).view(np.uint32) == want, (base, got)


def test_argument_errors_come_back_as_status_codes():
    lib = _abi.load_library()
    assert lib.pam_hip_pam_fwd(None, None, None, 16, 1.0, None) == -1
    assert b"null pointer" in lib.pam_hip_last_error()
    assert lib.pam_hip_pam_fwd(None, None, None, 0, 1.0, None) == 0          # empty input is fine
    assert lib.pam_hip_pam_matmul_fwd(None, 1, 1, None, 1, 1, None, 1, 1, -1, 4, 4, 1.0, None, 0, None) == -1
    assert lib.pam_hip_pam_matmul_fwd(None, 1, 1, None, 1, 1, None, 1, 1, 0, 4, 4, 1.0, None, 0, None) == 0
    c = _abi.gemm_plan(1, 12608, 768, 192)
    assert c % 32 == 0 and c >= 192
    c = _abi.gemm_plan(1, 192, 768, 12608)
    assert c % 32 == 0 and 128 <= c < 12608     # long k, few outputs: every tile's k range is cut into pieces of 128 k or more
    pieces = -(-12608 // c)
    assert _abi.load_library().pam_hip_gemm_workspace_bytes(1, 192, 768, 12608) == (64 << 10) + pieces * 36 * 64 * 64 * 4     # arrival words + a piece per unit
    assert _abi.load_library().pam_hip_gemm_workspace_bytes(1, 12608, 768, 192) == 0        # whole tiles: no scratch


class OracleKernels:
    """Same fourteen methods as the kernel object, computed by the CPU oracle on CPU tensors."""

    def __init__(self, oracle):
        self.o = oracle
        self.calls = []

    @staticmethod
    def _np(t):
        return t.detach().numpy()

    def _ret(self, a):
        return torch.from_numpy(np.array(a, dtype=np.float32, order="C"))      # keeps 0-d results 0-d

    def _off(self, offset):
        return None if offset == 1.0 else offset

    def pam_fwd(self, A, B, offset):
        self.calls.append(("pam_fwd", A.stride(), B.stride()))
        return self._ret(self.o.pam(self._np(A), self._np(B), self._off(offset)).reshape(A.shape))

    def pad_fwd(self, A, B, offset):
        return self._ret(self.o.pad(self._np(A), self._np(B), self._off(offset)).reshape(A.shape))

    def pam_bwd(self, A, B, dC, offset):
        return self._ret(self.o.pam_bwd(self._np(A), self._np(B), self._np(dC), self._off(offset)).reshape(A.shape))

    def pad_bwd(self, A, B, dC, offset):
        return self._ret(self.o.pad_bwd(self._np(A), self._np(B), self._np(dC), self._off(offset)).reshape(A.shape))

    def pa_exp_fwd(self, X, base, offset):
        return self._ret(self.o.pa_exp(self._np(X), base, self._off(offset)).reshape(X.shape))

    def pa_log_fwd(self, X, base, offset):
        return self._ret(self.o.pa_log(self._np(X), base, self._off(offset)).reshape(X.shape))

    def pa_exp_bwd(self, X, dY, base, offset):
        return self._ret(self.o.pa_exp_bwd(self._np(X), self._np(dY), base, self._off(offset)).reshape(X.shape))

    def pa_log_bwd(self, X, dY, base, offset):
        return self._ret(self.o.pa_log_bwd(self._np(X), self._np(dY), base, self._off(offset)).reshape(X.shape))

    def _mm(self, name, L, R, lrm, rrm, offset, mode=0, D=None):
        self.calls.append((name, tuple(L.stride()), tuple(R.stride()), lrm, rrm))
        # the flags must describe the strides they come with (pam/cuda_bindings.py:106-115)
        assert (L.stride()[-1] == 1) == lrm or L.stride()[-2] == 1
        assert (R.stride()[-1] == 1) == rrm or R.stride()[-2] == 1
        return self._ret(self.o.gemm(self._np(L), self._np(R), mode=mode, D=None if D is None else self._np(D),
                                     offset=self._off(offset)))

    def pam_matmul_fwd(self, A, B, arm, brm, offset):
        return self._mm("pam_matmul_fwd", A, B, arm, brm, offset)

    def pam_bmm_fwd(self, A, B, arm, brm, offset):
        return self._mm("pam_bmm_fwd", A, B, arm, brm, offset)

    def standard_matmul(self, A, B, arm, brm, offset):
        return self._mm("standard_matmul", A, B, arm, brm, offset, mode=1)

    def standard_bmm(self, A, B, arm, brm, offset):
        return self._mm("standard_bmm", A, B, arm, brm, offset, mode=1)

    def pam_matmul_bwd(self, L, R, M, lrm, rrm, delta_L, offset):
        return self._mm("pam_matmul_bwd", L, R, lrm, rrm, offset, mode=2 if delta_L else 3, D=M)

    def pam_bmm_bwd(self, L, R, M, lrm, rrm, delta_L, offset):
        return self._mm("pam_bmm_bwd", L, R, lrm, rrm, offset, mode=2 if delta_L else 3, D=M)


@pytest.fixture()
def fake(oracle, monkeypatch):
    k = OracleKernels(oracle)
    monkeypatch.setattr(cuda_bindings, "cuda_kernels", k)
    return k


def _t(shape, seed, grad=True):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(*shape, generator=g).requires_grad_(grad)


def test_elementwise_autograd_formulas(fake, oracle):
    A, B = _t((7, 5), 1), _t((7, 5), 2)
    dY = _t((7, 5), 3, grad=False)
    for off in (None, 1.0552):
        for approx in (True, False, (True, False), (False, True)):
            A.grad = B.grad = None
            cuda_bindings.pam(A, B, offset=off, approx_bwd=approx).backward(dY)
            ap = (approx, approx) if isinstance(approx, bool) else approx
            a, b, d = A.detach().numpy(), B.detach().numpy(), dY.numpy()
            want_a = oracle.pam(d, b, off) if ap[0] else oracle.pam_bwd(a, b, d, off)      # pam/cuda_bindings.py:47-55
            want_b = oracle.pam(d, a, off) if ap[1] else oracle.pam_bwd(b, a, d, off)
            assert_same_bits(A.grad.numpy(), want_a, f"dA {off} {approx}")
            assert_same_bits(B.grad.numpy(), want_b, f"dB {off} {approx}")
    # division: the GPU flavour of the formulas (pam/cuda_bindings.py:86-95)
    A.grad = B.grad = None
    cuda_bindings.pad(A, B, approx_bwd=True).backward(dY)
    a, b, d = A.detach().numpy(), B.detach().numpy(), dY.numpy()
    assert_same_bits(A.grad.numpy(), oracle.pam(oracle.pad(np.ones_like(b), b), d), "pad dA approx")
    assert_same_bits(B.grad.numpy(), -oracle.pam(oracle.pad(oracle.pad(a, b), b), d), "pad dB approx")
    A.grad = B.grad = None
    cuda_bindings.pad(A, B, approx_bwd=False).backward(dY)
    assert_same_bits(A.grad.numpy(), oracle.pam_bwd(a, oracle.pad(np.ones_like(b), b), d), "pad dA exact")
    assert_same_bits(B.grad.numpy(), oracle.pad_bwd(a, b, d), "pad dB exact")


def test_broadcast_and_scalars(fake, oracle):
    A = _t((4, 3), 5)
    out = cuda_bindings.pam(A, 2.0)
    assert_same_bits(out.detach().numpy(), A.detach().numpy() * 2.0, "x * 2")
    out.sum().backward()
    assert A.grad.shape == A.shape
    row = _t((3,), 6)
    out = cuda_bindings.pam(A, row, approx_bwd=True)
    out.backward(torch.ones_like(out))
    assert row.grad.shape == (3,)                 # autograd sums over the broadcast dimension
    assert_same_bits(row.grad.numpy(), oracle.pam(np.ones((4, 3), np.float32), A.detach().numpy()).sum(0), "broadcast grad")


def test_exp_log_autograd_formulas(fake, oracle):
    X = _t((6, 4), 7); dY = _t((6, 4), 8, grad=False)
    x, d = X.detach().numpy(), dY.numpy()
    for base in (math.e, 2.0, 10.0):
        X.grad = None
        y = cuda_bindings.pa_exp(X, base=base, approx_bwd=True); y.backward(dY)
        grad = oracle.pa_exp(x, base)
        if base != math.e:
            grad = oracle.pam(grad, np.full_like(x, math.log(base)))
        assert_same_bits(X.grad.numpy(), oracle.pam(grad, d), f"exp approx {base}")        # pam/cuda_bindings.py:228-235
        X.grad = None
        cuda_bindings.pa_exp(X, base=base, approx_bwd=False).backward(dY)
        assert_same_bits(X.grad.numpy(), oracle.pa_exp_bwd(x, d, base), f"exp exact {base}")
        Xp = X.detach().abs().requires_grad_()
        cuda_bindings.pa_log(Xp, base=base, approx_bwd=True).backward(dY)
        grad = oracle.pad(d, Xp.detach().numpy())
        if base != math.e:
            grad = oracle.pad(grad, np.full_like(x, math.log(base)))
        assert_same_bits(Xp.grad.numpy(), grad, f"log approx {base}")                    # pam/cuda_bindings.py:268-272
    assert_same_bits(cuda_bindings.pa_exp2(X).detach().numpy(), oracle.pa_exp(x, 2.0), "exp2")
    assert_same_bits(cuda_bindings.pa_log2(X.detach().abs()).numpy(), oracle.pa_log(np.abs(x), 2.0), "log2")


def test_check_row_major():
    t = torch.zeros(4, 6)
    assert cuda_bindings.check_row_major(t, 2)[1] is True
    v, rm = cuda_bindings.check_row_major(t.T, 2)
    assert rm is False and v.data_ptr() == t.data_ptr()              # a transposed view is passed on, not copied
    s = torch.zeros(4, 12)[:, ::2]
    c, rm = cuda_bindings.check_row_major(s, 2)
    assert rm is True and c.is_contiguous() and c.data_ptr() != s.data_ptr()
    with pytest.raises(ValueError):
        cuda_bindings.check_row_major(t, 3)
    q = torch.zeros(8, 6, 4).transpose(0, 1)                          # fairseq-style (B*H, T, D) view of (T, B*H, D)
    assert cuda_bindings.check_row_major(q, 3)[1] is True and cuda_bindings.check_row_major(q.transpose(1, 2), 3)[1] is False


def test_matmul_autograd_uses_views(fake, oracle):
    A = _t((9, 6), 9); Bt = _t((5, 6), 10)                 # B given as W.T, the nn.Linear case
    dY = _t((9, 5), 11, grad=False)
    a, b, d = A.detach().numpy(), Bt.detach().numpy().T, dY.numpy()
    Y = cuda_bindings.pam_matmul(A, Bt.T, approx_bwd=True)
    assert_same_bits(Y.detach().numpy(), oracle.gemm(a, b), "forward")
    Y.backward(dY)
    assert_same_bits(A.grad.numpy(), oracle.gemm(d, b.T), "dA = dY B^T")               # pam/cuda_bindings.py:155
    assert_same_bits(Bt.grad.numpy().T, oracle.gemm(a.T, d), "dB = A^T dY")            # pam/cuda_bindings.py:161
    fwd = [c for c in fake.calls if c[0] == "pam_matmul_fwd"]
    assert fwd[0][1:] == ((6, 1), (1, 6), True, False)       # X row-major, W.T column-major view
    assert fwd[1][1:] == ((5, 1), (6, 1), True, True)        # dY row-major, (W.T).mT = W row-major: no copy
    assert fwd[2][1:] == ((1, 6), (5, 1), False, True)       # X.mT column-major view, dY row-major
    A.grad = Bt.grad = None
    cuda_bindings.pam_matmul(A, Bt.T, approx_bwd=False).backward(dY)
    assert_same_bits(A.grad.numpy(), oracle.gemm(d, b.T, mode=oracle.MODE_BWD_DELTA_L, D=a), "exact dA")
    assert_same_bits(Bt.grad.numpy().T, oracle.gemm(a.T, d, mode=oracle.MODE_BWD_DELTA_R, D=b), "exact dB")
    # batched, tuple flag, standard product
    P, V = _t((3, 7, 4), 12), _t((3, 4, 6), 13); dO = _t((3, 7, 6), 14, grad=False)
    cuda_bindings.pam_bmm(P, V, approx_bwd=(True, False)).backward(dO)
    p, v, do = P.detach().numpy(), V.detach().numpy(), dO.numpy()
    assert_same_bits(P.grad.numpy(), oracle.gemm(do, np.swapaxes(v, 1, 2)), "bmm dA approx")
    assert_same_bits(V.grad.numpy(), oracle.gemm(np.swapaxes(p, 1, 2), do, mode=oracle.MODE_BWD_DELTA_R, D=v), "bmm dB exact")
    S = cuda_bindings.standard_matmul(A.detach(), Bt.detach().T, offset=1.5, approx_bwd=True)
    assert np.allclose(S.numpy(), a @ b, rtol=1e-5, atol=1e-6)


def test_op_library_surface(fake):
    for name in ("mul", "div", "exp", "exp2", "log", "log2", "pow", "matmul", "bmm", "linear", "Linear"):
        assert hasattr(pam_amd, name)
    x = torch.randn(3, 4)
    with pytest.raises(RuntimeError, match="GPU only"):
        pam_ops.mul(x, x)                                   # no CPU fallback in this package
    with pytest.raises(NotImplementedError):
        pam_ops.matmul(x, x.T, use_kernel=False)
    with pytest.raises(AssertionError):
        pam_ops.bmm(torch.zeros(2, 3, 4), torch.zeros(3, 4, 5))
    lin = pam_amd.Linear(8, 3, offset=1.0552, approx_bwd=True)
    ref = torch.nn.Linear(8, 3)
    lin.load_state_dict(ref.state_dict())                   # same parameters as torch.nn.Linear (pam/pam_ops.py:259-264)
    assert set(lin.state_dict()) == set(ref.state_dict())
    assert "offset=1.05520" in repr(lin) and "approx_bwd=True" in repr(lin) and repr(lin).startswith("pam.Linear")


def test_kernel_object_rejects_host_tensors():
    k = _abi.HipKernels()
    x = torch.randn(4, 4)
    with pytest.raises(RuntimeError, match="CUDA tensor"):           # CHECK_CUDA, pam/cuda_kernels.cu:8
        k.pam_fwd(x, x, 1.0)
    with pytest.raises(RuntimeError, match="CUDA tensor"):
        k.pam_matmul_fwd(x, x, True, True, 1.0)


def test_bench_refuses_more_than_one_gpu():
    """The benchmark measures one GPU; asking for more ends with a message instead of a silent single-GPU run."""
    import pathlib
    import subprocess
    import sys
    root = pathlib.Path(__file__).resolve().parents[1]
    res = subprocess.run([sys.executable, str(root / "bench.py"), "--gpus", "2"], capture_output=True, text=True, timeout=120)
    assert res.returncode != 0 and "one GPU" in res.stderr and res.stdout.strip() == ""


@pytest.mark.gpu
@pytest.mark.parametrize("op", ["linear", "matmul", "bmm", "softmax", "layer_norm"])
def test_nodes_keep_autograds_rules(op):
    """The ops whose autograd nodes are in C++: saved-tensor hooks see their tensors, a tensor changed in place after the
    forward pass is an error, gradients come only for what asks for one, a gradient that is differentiated again keeps
    the graph of its ordinary sums, and a flag that is none only fails a backward pass."""
    torch.manual_seed(0)
    new = lambda *shape: torch.randn(*shape, device="cuda")
    inputs = {"linear": [new(33, 20), new(24, 20), new(24)], "matmul": [new(33, 20), new(20, 24)], "bmm": [new(3, 9, 20), new(3, 20, 8)],
              "softmax": [new(5, 37)], "layer_norm": [new(5, 6, 40), new(40), new(40)]}[op]
    call = {"linear": pam_amd.linear, "matmul": pam_amd.matmul, "bmm": pam_amd.bmm,
            "softmax": lambda x, **kw: pam_amd.softmax(x, dim=-1, **kw),
            "layer_norm": lambda x, w, b, **kw: pam_amd.layer_norm(x, 40, w, b, **kw)}[op]
    leaves = [t.clone().requires_grad_() for t in inputs]
    y = call(*leaves, approx_bwd=True)
    dy = torch.randn_like(y)
    want = torch.autograd.grad(y, leaves, dy)
    assert all(g.shape == t.shape for g, t in zip(want, leaves)) and not call(*inputs).requires_grad

    seen = []
    def pack(t):
        seen.append(t.shape)
        return t.cpu()
    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.cuda()):
        y = call(*leaves, approx_bwd=True)
    assert seen and all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(y, leaves, dy), want))

    for i in range(len(inputs)):                                        # one gradient at a time
        some = [t.clone().requires_grad_(j == i) for j, t in enumerate(inputs)]
        g, = torch.autograd.grad(call(*some, approx_bwd=True), [some[i]], dy)
        assert torch.equal(g, want[i])

    y = call(*leaves, approx_bwd=True)
    with torch.no_grad():
        leaves[0].mul_(1.0)
    with pytest.raises(RuntimeError, match="inplace operation"):
        torch.autograd.grad(y, leaves, dy)

    if op in ("linear", "layer_norm"):                                    # the bias gradient is a plain sum of dy
        dyr = dy.clone().requires_grad_()
        grads = torch.autograd.grad(call(*leaves, approx_bwd=True), leaves, dyr, create_graph=True)
        again, = torch.autograd.grad(grads[2].sum(), dyr)
        assert torch.equal(again, torch.ones_like(dy))

    y = call(*leaves, approx_bwd=None)
    with pytest.raises(TypeError):
        torch.autograd.grad(y, leaves, dy)
    if op in ("matmul", "bmm"):
        with pytest.raises(TypeError):
            call(*[t.double() for t in inputs])


@pytest.mark.gpu
def test_nodes_on_threads_and_streams():
    """Products that cut their tiles, from several threads on streams of their own at once: each as alone (every stream has
    its own scratch)."""
    import threading
    torch.manual_seed(1)
    data = [[torch.randn(300, 4096, device="cuda"), torch.randn(4096, 100 + 30 * i, device="cuda")] for i in range(4)]
    want = [pam_amd.matmul(a, b) for a, b in data]
    torch.cuda.synchronize()
    bad = []
    def work(i):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for _ in range(10):
                if not torch.equal(pam_amd.matmul(*data[i]), want[i]):
                    bad.append(i)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


@pytest.mark.parametrize("shape,exact,want", [
    # (1024 work-groups are resident: four on each of 256 compute units)
    ((1, 96, 128, 64), 0, 0), ((1, 512, 4096, 64), 0, 0),                       # a round of at most two per compute unit: nothing to even out
    ((1, 2112, 1024, 96), 0, 1), ((1, 4096, 1024, 512), 0, 1), ((192, 197, 64, 197), 0, 1),     # more than half a round
    ((1, 4352, 1024, 96), 0, 0), ((128, 128, 576, 1024), 0, 0), ((128, 128, 576, 1024), 1, 0),  # one more per compute unit behind a full round or two
    ((1, 12608, 768, 192), 0, 1), ((1, 12608, 768, 192), 1, 0),                 # two more behind: whole tiles, and deep enough
    ((1, 12544 + 63, 768, 192), 0, 0), ((192, 197, 133, 64), 0, 0),             # ragged ones, shallow ones
    ((51, 128, 900, 864), 0, 1), ((704, 64, 130, 224), 0, 0),                   # ragged, but deep; ragged and not deep
    ((128, 64, 1024, 1152), 0, 1), ((128, 64, 1024, 1152), 1, 1),               # two full rounds
    ((1, 192, 768, 12608), 0, 1), ((1, 192, 768, 12608), 1, 1),                 # 57 pieces of 36 tiles: two rounds and four short units
    ((1, 364, 233, 13642), 0, 0),                                               # 43 pieces of 24 tiles: a round and eight units of 0.7 the length
    ((512, 128, 128, 64), 0, 0), ((1, 8192, 1024, 128), 1, 0), ((1, 8192, 1024, 256), 1, 1), ((1, 16384, 1024, 256), 1, 0), ((1, 16384, 1024, 320), 1, 1)])
def test_priorities_fall_only_where_the_last_round_fills_the_chip(shape, exact, want):
    assert _abi.load_library().pam_hip_gemm_priority_steps(*shape, exact) == want


@pytest.mark.parametrize("shape,kind,schedule,steps", [
    ((192, 197, 197, 64), 0, (16, 100, 40, 1920), 1), ((192, 197, 197, 64), 1, (16, 64, 64, 3072), 0),      # a mostly full second round; the exact gradient
    ((181, 89, 89, 64), 0, (16, 64, 64, 724), 1), ((43, 211, 211, 64), 0, (16, 64, 64, 688), 1),            # three on the fullest compute unit either way
    ((165, 196, 32, 196), 0, (32, 64, 64, 660), 1), ((600, 100, 30, 60), 0, (16, 100, 32, 600), 1),         # narrow results, resident and beyond
    ((1, 50432, 32, 64), 0, (16, 128, 32, 394), 0), ((1, 4096, 1024, 512), 0, (32, 64, 64, 1024), 1)])     # one per compute unit and a half; whole tiles
def test_schedules_are_those_of_the_launch(shape, kind, schedule, steps):
    """What the library reports of a product is what it launches, freely shaped tiles among them."""
    assert _abi.gemm_schedule(*shape, kind) == schedule
    assert _abi.load_library().pam_hip_gemm_priority_steps(*shape, kind) == steps


@pytest.mark.parametrize("shape,pieces,fullest", [((1, 192, 192, 12608), 57, 3), ((110, 71, 71, 128), 1, 2), ((47, 244, 128, 244), 2, 3), ((1, 77, 3983, 594), 4, 2),
                                                  ((8, 192, 144, 768), 6, 2), ((4, 64, 841, 1152), 9, 2), ((1, 192, 768, 12608), 57, 9),
                                                  ((1, 644, 864, 480), 3, 2), ((1, 3623, 140, 560), 4, 3), ((19, 64, 576, 576), 4, 3)])
def test_plans_price_the_fullest_compute_unit(shape, pieces, fullest):
    """Products that evenly counted units put on a fuller compute unit than the plan that is measured the faster one."""
    assert -(-shape[3] // _abi.gemm_plan(*shape)) == pieces and -(-_abi.gemm_schedule(*shape)[3] // 256) == fullest


@pytest.mark.parametrize("shapes", [[(1, 64, 64, k) for k in (8192, 16384, 32768, 65536, 98304)],
                                    [(1, m, n, k) for a, b in ((192, 768), (192, 192), (768, 192)) for m, n, k in ((12608, b, a), (12608, a, b), (a, b, 12608))]])
def test_plans_of_a_models_sizes_are_kept_side_by_side(shapes):
    """Sizes that are multiples of 32 do not push each other's plans out: asking for several in turn takes hardly longer than
    asking for one (found anew each time, the first ones take thirty times as long)."""
    import time
    ask = _abi.load_library().pam_hip_gemm_workspace_bytes
    def fastest(shapes):
        best = math.inf
        for _ in range(20):
            start = time.perf_counter()
            for i in range(360):
                ask(*shapes[i % len(shapes)])
            best = min(best, time.perf_counter() - start)
        return best
    assert fastest(shapes) < 1.6 * fastest(shapes[:1])


def test_forced_k_tiles_hold_for_every_product():
    """The tuning hook's depth is taken by products and convolutions alike, whatever the rule for their sizes is."""
    lib, shape = _abi.load_library(), (100, 64, 1024, 144)
    assert _abi.gemm_schedule(*shape, 2)[0] == 16
    try:
        for depth in (16, 32):
            lib.pam_hip_set_tuning(depth, 1)
            assert [_abi.gemm_schedule(*shape, kind)[0] for kind in (0, 1, 2)] == [depth] * 3
    finally:
        lib.pam_hip_set_tuning(0, 0)


@pytest.mark.gpu
def test_other_threads_run_while_a_launch_waits():
    """Behind one long product thousands of small ones fill the launch queue, and the next call waits for it: other
    Python threads go on meanwhile."""
    import threading
    import time
    a, b = torch.ones(16384, 65536, device="cuda"), torch.ones(65536, 16384, device="cuda")
    small = torch.ones(1, 1, device="cuda")
    pam_amd.matmul(a[:64], b[:, :64])
    pam_amd.matmul(small, small)
    torch.cuda.synchronize()
    gaps, stop = [0.0], threading.Event()
    def tick():
        last = time.perf_counter()
        while not stop.is_set():
            time.sleep(1e-3)
            now = time.perf_counter()
            gaps.append(now - last)
            last = now
    thread = threading.Thread(target=tick)
    thread.start()
    began = time.perf_counter()
    pam_amd.matmul(a, b)
    for _ in range(25000):
        pam_amd.matmul(small, small)
    queued = time.perf_counter() - began
    torch.cuda.synchronize()
    stop.set()
    thread.join()
    print(f"queued in {queued:.2f} s, longest gap {max(gaps):.3f} s")
    assert max(gaps) < 0.2, (queued, max(gaps))


@pytest.mark.gpu
@pytest.mark.parametrize("how", ["object", "method"])
@pytest.mark.parametrize("approx", [True, False, (True, False)])
def test_swapped_kernel_objects_are_called(monkeypatch, how, approx):
    """Another object in place of `fused.row_kernels` or `cuda_bindings.cuda_kernels`, or a method replaced on the one that is
    there, computes the ops that go through it, forward and backward; one that passes the calls on gives the same bits."""
    from pam_amd import fused
    torch.manual_seed(2)
    calls = []

    class Recorder:                        # the methods as callers know them, without optional arguments of the package's own
        def __init__(self, kernels):
            self.kernels = kernels
        def __getattr__(self, name):
            method = getattr(self.kernels, name)
            def call(*args):
                assert name != "logsumexp_fwd" or len(args) == 4
                calls.append(name)
                return method(*args)
            return call

    x, w, b = (torch.randn(*s, device="cuda") for s in ((6, 37, 40), (40,), (40,)))
    wl, bl = torch.randn(24, 40, device="cuda"), torch.randn(24, device="cuda")
    ops = {
        "softmax": (lambda x: pam_amd.softmax(x, dim=-1, approx_bwd=approx), (x,), fused, ["softmax_fwd", "softmax_bwd"]),
        "log_softmax": (lambda x: pam_amd.log_softmax(x, dim=-1, approx_bwd=approx), (x,), fused, ["logsumexp_fwd", "logsumexp_bwd"]),
        "layer_norm": (lambda x, w, b: pam_amd.layer_norm(x, 40, w, b, approx_bwd=approx), (x, w, b), fused, ["layer_norm_fwd", "layer_norm_bwd"]),
        "linear": (lambda x, w, b: pam_amd.linear(x, w, b, approx_bwd=approx), (x, wl, bl), cuda_bindings, ["pam_matmul_fwd", "pam_matmul_bwd"]),
        "matmul": (lambda x, w: pam_amd.matmul(x, w, approx_bwd=approx), (x[0], wl.t()), cuda_bindings, ["pam_matmul_fwd", "pam_matmul_bwd"]),
    }
    for op, (f, inputs, module, names) in ops.items():
        def run():
            leaves = [t.detach().clone().requires_grad_() for t in inputs]
            y = f(*leaves)
            return [y, *torch.autograd.grad(y, leaves, torch.linspace(-1, 1, y.numel(), device="cuda").view(y.shape))]
        want = run()
        assert not calls
        holder = "row_kernels" if module is fused else "cuda_kernels"
        with monkeypatch.context() as m:
            recorder = Recorder(type(getattr(module, holder))())
            if how == "object":
                m.setattr(module, holder, recorder)
            else:
                # (in the object's own dictionary: setattr would leave the class's methods there when it is undone, and every later
                # test of the process would run the autograd functions in Python)
                for name in names:
                    m.setitem(vars(getattr(module, holder)), name, getattr(recorder, name))
            got = run()
        expected = set(names)
        if op in ("linear", "matmul"):
            expected = {"pam_matmul_fwd"} if approx is True else {"pam_matmul_bwd"} if approx is False and op == "linear" else set(names)
        assert set(calls) == expected, (op, calls)
        calls.clear()
        for a, c in zip(got, want):
            assert torch.equal(a, c), op
    assert not calls and run() is not None and not calls
    assert not vars(fused.row_kernels) and not vars(cuda_bindings.cuda_kernels)


def test_build_stamp_covers_what_the_host_module_is_built_on(monkeypatch, tmp_path):
    """The built files count as current for this torch and these flags, wherever the tree lies, and for no others."""
    from pam_amd import build as builder
    assert builder.built_hash() == builder.source_hash()
    host_hash, flags = builder.host_hash(), builder._host_flags()
    with monkeypatch.context() as m:
        m.setattr(builder, "LIB", tmp_path / "elsewhere" / "libpam_hip.so")
        assert builder.host_hash() == host_hash
    for what in ("torch", "flags", "link"):
        with monkeypatch.context() as m:
            if what == "torch":
                m.setattr(torch, "__version__", "0.0")
            else:
                m.setattr(builder, "_host_flags", lambda: (flags[0] + ["-O1"], flags[1]) if what == "flags" else (flags[0], flags[1] + ["-lm"]))
            assert builder.built_hash() is None
    assert builder.built_hash() == builder.source_hash()


def test_build_links_the_library_without_the_host_modules_needs(monkeypatch, tmp_path):
    """Where g++ or torch's headers are missing the library is still linked (a program in C needs no more), the failure
    is reported, and no host module of another build stays beside it."""
    from pam_amd import build as builder
    ran = []
    def run(cmd, verbose):
        ran.append(cmd)
        if cmd[0] == "g++":
            raise RuntimeError("g++ failed")
    monkeypatch.setattr(builder, "_run", run)
    monkeypatch.setattr(builder, "LIB", tmp_path / "libpam_hip.so")
    monkeypatch.setattr(builder, "HOST", tmp_path / "_pam_host.so")
    builder.HOST.write_text("an older one")
    with pytest.raises(RuntimeError, match="g\\+\\+"):
        builder.build()
    assert any("-shared" in cmd and str(builder.LIB) in cmd for cmd in ran) and not builder.HOST.exists()


@pytest.mark.gpu
@pytest.mark.filterwarnings("ignore::torch.jit.TracerWarning")
@pytest.mark.parametrize("op", ["linear", "matmul", "bmm", "softmax", "log_softmax", "layer_norm"])
def test_traced_functions_compute_on_new_inputs(op):
    """torch.jit.trace records the ops: a traced function gives on other inputs, forward and backward, what the ops give."""
    torch.manual_seed(4)
    new = lambda *shape: torch.randn(*shape, device="cuda")
    w, b, right = new(24, 40), new(24), new(3, 40, 7)
    f = {"linear": lambda x: pam_amd.linear(x, w, b, approx_bwd=True), "matmul": lambda x: pam_amd.matmul(x[0], w.t(), approx_bwd=True),
         "bmm": lambda x: pam_amd.bmm(x, right, approx_bwd=True), "softmax": lambda x: pam_amd.softmax(x, dim=-1, approx_bwd=True),
         "log_softmax": lambda x: pam_amd.log_softmax(x, dim=-1, approx_bwd=True),
         "layer_norm": lambda x: pam_amd.layer_norm(x, 40, w[0], w[1], approx_bwd=True)}[op]
    for grad in (False, True):
        traced = torch.jit.trace(f, (new(3, 6, 40).requires_grad_(grad),), check_trace=False)
        x = new(3, 6, 40)
        assert torch.equal(traced(x), f(x))
        if grad:
            x = x.requires_grad_()
            dy = torch.randn_like(f(x))
            assert torch.equal(torch.autograd.grad(traced(x), x, dy)[0], torch.autograd.grad(f(x), x, dy)[0])


@pytest.mark.gpu
def test_rows_of_a_tensor_subclass_keep_their_class():
    """softmax, log_softmax and layer_norm of a subclass are of that class, of a Parameter ordinary tensors."""
    class Marked(torch.Tensor):
        pass
    x, w = torch.randn(6, 40, device="cuda"), torch.randn(40, device="cuda")
    for f in (lambda t: pam_amd.softmax(t, dim=-1), lambda t: pam_amd.log_softmax(t, dim=-1), lambda t: pam_amd.layer_norm(t, 40, w, w)):
        got = f(x.as_subclass(Marked))
        assert type(got) is Marked and torch.equal(got.as_subclass(torch.Tensor), f(x))
        assert type(f(torch.nn.Parameter(x))) is torch.Tensor


@pytest.mark.gpu
@pytest.mark.parametrize("op", ["linear", "matmul", "softmax", "layer_norm"])
def test_unusual_flags_and_offsets_are_taken_or_refused_where_they_were(op):
    """approx_bwd is unpacked in the backward pass only: a list or a tensor of two is a pair, anything else that is no flag
    fails there, with the error of the unpacking, and not in a forward pass.  An offset is whatever float() takes."""
    torch.manual_seed(6)
    x, w, b = (torch.randn(*s, device="cuda") for s in ((6, 40), (24, 40), (24,)))
    f = {"linear": lambda x, **kw: pam_amd.linear(x, w, b, **kw), "matmul": lambda x, **kw: pam_amd.matmul(x, w.t(), **kw),
         "softmax": lambda x, **kw: pam_amd.softmax(x, dim=-1, **kw), "layer_norm": lambda x, **kw: pam_amd.layer_norm(x, 40, w[0], w[1], **kw)}[op]
    def gradient(**kw):
        leaf = x.clone().requires_grad_()
        y = f(leaf, **kw)
        return torch.autograd.grad(y, leaf, torch.linspace(-1, 1, y.numel(), device="cuda").view(y.shape))[0]
    pair = gradient(approx_bwd=(True, False))
    assert torch.equal(gradient(approx_bwd=[True, False]), pair)
    if op in ("linear", "matmul"):
        assert torch.equal(gradient(approx_bwd=torch.tensor([True, False])), pair)
    for flag, error in ((None, TypeError), (1, TypeError), (np.bool_(True), TypeError), ((True,), ValueError), ((True,) * 3, ValueError)):
        assert torch.equal(f(x, approx_bwd=flag), f(x))
        with pytest.raises(error):
            gradient(approx_bwd=flag)
    want = f(x, offset=1.0552)
    for offset in (np.float64(1.0552), np.float32(1.0552), torch.tensor(1.0552)):
        assert torch.equal(f(x, offset=offset), want)
    with pytest.raises(ValueError):
        f(x, offset="x")


@pytest.mark.gpu
def test_refusals_say_what_they_said():
    """The checks of the products in C++: kinds of error, names, types and shapes as Python prints them."""
    K, x, w = _abi.HipKernels(), torch.randn(6, 40, device="cuda"), torch.randn(24, 40, device="cuda")
    b = torch.randn(24, device="cuda")
    for call, error, text in (
            (lambda: K.pam_matmul_fwd(x, w, True, True, 1.0), ValueError, r"pam_matmul_fwd: shapes \(6, 40\) and \(24, 40\) do not multiply"),
            (lambda: K.pam_bmm_fwd(x, w.t(), True, True, 1.0), ValueError, "pam_bmm_fwd: expected 3-D operands"),
            (lambda: K.standard_matmul(x[None], w.t(), True, True, 1.0), ValueError, "standard_matmul: expected 2-D operands"),
            (lambda: K.pam_bmm_fwd(x.expand(2, 6, 40), w.t().expand(3, 40, 24), True, True, 1.0), ValueError, r"shapes \(2, 6, 40\) and \(3, 40, 24\) do not"),
            (lambda: K.pam_matmul_bwd(x, w.t(), None, True, True, True, 1.0), TypeError, "the forward operand is missing"),
            (lambda: K.pam_matmul_bwd(x, w.t(), x, True, True, True, 1.0), ValueError, "third operand must have the shape of the result"),
            (lambda: pam_amd.matmul(x.half(), w.t()), TypeError, "PAM kernels compute in float32, got torch.float16"),
            (lambda: pam_amd.linear(x, w[:, :39], b), ValueError, r"linear_fwd: shapes \(6, 40\) and \(39, 24\) do not multiply"),
            (lambda: pam_amd.linear(x, w, b[:23]), ValueError, "linear_fwd: bias must be contiguous with one value per output column"),
            (lambda: pam_amd.matmul(x, w.t().cpu()), RuntimeError, "argument must be a CUDA tensor")):
        with pytest.raises(error, match=text):
            call()


@pytest.mark.gpu
@pytest.mark.parametrize("offset", [None, 1.0552])
@pytest.mark.parametrize("approx", [True, False, (True, False), (False, True)])
def test_elementwise_and_log_softmax_nodes_equal_the_autograd_functions(offset, approx):
    """Results, gradients (also of an expanded upstream gradient, and of one operand alone) and refusals of the nodes in C++
    are those of the autograd functions in Python."""
    import math
    from pam_amd import cuda_bindings as cb, fused
    g = torch.Generator(device="cuda").manual_seed(1)
    a0, b0 = torch.randn(37, 129, generator=g, device="cuda"), torch.randn(37, 129, generator=g, device="cuda")
    b0[0, :5] = torch.tensor([0.0, 1e-40, 3e38, -1e-30, -0.0])
    pos = a0.abs() + 1e-3
    kw = dict(offset=offset, approx_bwd=approx)
    pairs = [(lambda a, b: pam_amd.mul(a, b, **kw), lambda a, b: cb.pam_autograd.apply(a, b, offset, approx), (a0, b0)),
             (lambda a, b: pam_amd.div(a, b, **kw), lambda a, b: cb.pad_autograd.apply(a, b, offset, approx), (a0, b0))]
    for base in (math.e, 2.0, 10):
        pairs += [(lambda a, base=base: cb.pa_exp(a, base=base, **kw), lambda a, base=base: cb.pa_exp_autograd.apply(a, base, offset, approx), (a0,)),
                  (lambda a, base=base: cb.pa_log(a, base=base, **kw), lambda a, base=base: cb.pa_log_autograd.apply(a, base, offset, approx), (pos,))]
    pairs += [(lambda a, p=p: pam_amd.pow(a, p, **kw), lambda a, p=p: fused.pow_autograd.apply(a, p, offset, approx), (pos,)) for p in (0.5, 3)]
    rows = lambda a: a.reshape(-1, a.shape[-1])
    pairs += [(lambda a: pam_amd.log_softmax(a, dim=-1, **kw), lambda a: fused.logsumexp_autograd.apply(rows(a), offset, approx, True, True).view(a.shape), (a0,)),
              (lambda a: pam_amd.logsumexp(a, -1, **kw), lambda a: fused.logsumexp_autograd.apply(rows(a), offset, approx, False, True).view(a.shape[:-1]), (a0,)),
              (lambda a: pam_amd.logsumexp(a, -1, keepdim=True, **kw), lambda a: fused.logsumexp_autograd.apply(rows(a), offset, approx, False, True).view(a.shape[:-1] + (1,)), (a0,))]
    same = lambda x, y: x.shape == y.shape and torch.equal(x.nan_to_num(5.0, 6.0, 7.0), y.nan_to_num(5.0, 6.0, 7.0))
    for node, function, values in pairs:
        makes = [lambda t: t.clone(), lambda t: t.view(37, 1, 129).clone(), lambda t: torch.zeros(129, 37, device="cuda").t().copy_(t)]
        for make in makes[:2] if (node, function, values) in pairs[-3:] else makes:      # (rows that are not contiguous are a chain of ops)
            mine, theirs = [make(v).requires_grad_() for v in values], [make(v).requires_grad_() for v in values]
            y, want = node(*mine), function(*[t.contiguous() for t in theirs])
            assert same(y, want) and y.requires_grad and torch.equal(node(*[t.detach() for t in mine]).nan_to_num(5.0), y.detach().nan_to_num(5.0))
            for up in (torch.randn(y.shape, generator=g, device="cuda"), torch.full((1,), 0.7, device="cuda").expand(y.shape)):
                got = torch.autograd.grad(y, mine, up, retain_graph=True)
                assert all(same(p, q) for p, q in zip(got, torch.autograd.grad(want, theirs, up, retain_graph=True)))
                assert same(torch.autograd.grad(y, mine[-1], up, retain_graph=True)[0], got[-1])
            if len(mine) == 2:                              # one gradient wanted, then broadcast operands and numbers
                one = node(mine[0], values[1].view(mine[0].shape))
                assert same(torch.autograd.grad(one.sum(), mine[0])[0], torch.autograd.grad(want.sum(), theirs[0], retain_graph=True)[0])
                assert same(node(mine[0], values[1][:1, :1].expand(37, 129).reshape(mine[0].shape)), node(mine[0], values[1][0, 0]))
                assert same(node(mine[0], 1.5), node(mine[0], torch.full_like(mine[0], 1.5)))
    leaf = pos.clone().requires_grad_()
    for y in (pam_amd.mul(leaf, leaf, **kw), pam_amd.div(leaf, leaf, **kw), pam_amd.exp(leaf, **kw), pam_amd.log(leaf, **kw), pam_amd.pow(leaf, 0.5, **kw),
              pam_amd.log_softmax(leaf, dim=-1, **kw), pam_amd.logsumexp(leaf.view(1, -1), -1, keepdim=True, **kw).grad_fn.next_functions[0][0]):
        assert "Node" in (y if not isinstance(y, torch.Tensor) else y.grad_fn).name()      # (not an autograd function in Python)
    with pytest.raises(TypeError, match="float32"):
        pam_amd.mul(a0.double(), b0.double(), **kw)
    for bad in (float("inf"), float("nan")):
        x = a0.clone(); x[3, 4] = bad
        for op in (pam_amd.log_softmax, pam_amd.logsumexp):
            with pytest.raises(AssertionError):
                op(x, -1, **kw)
    assert torch.equal(pam_amd.log_softmax(a0, -1, **kw), pam_amd.log_softmax(a0, -1, **kw))      # (the word was cleared)


@pytest.mark.gpu
@pytest.mark.parametrize("op", ["mul", "div", "exp", "log", "pow", "softmax", "logsumexp", "log_softmax", "layer_norm"])
@pytest.mark.parametrize("approx", [True, False])
def test_saved_tensors_come_back_from_hooks_in_any_layout(op, approx):
    """Hooks may return other strides for a saved tensor, which give the same gradients; one of another type, size or device
    is refused before a kernel sees it."""
    torch.manual_seed(8)
    kw = dict(approx_bwd=approx)
    f = {"mul": lambda a, b: pam_amd.mul(a, b, **kw), "div": lambda a, b: pam_amd.div(a, b, **kw), "exp": lambda a, b: pam_amd.exp(a, **kw),
         "log": lambda a, b: pam_amd.log(a, **kw), "pow": lambda a, b: pam_amd.pow(a, 0.5, **kw), "softmax": lambda a, b: pam_amd.softmax(a, dim=-1, **kw),
         "logsumexp": lambda a, b: pam_amd.logsumexp(a, -1, **kw), "log_softmax": lambda a, b: pam_amd.log_softmax(a, dim=-1, **kw),
         "layer_norm": lambda a, b: pam_amd.layer_norm(a, 40, b[0], b[1], **kw)}[op]
    a, b = (torch.rand(24, 40, device="cuda").add_(0.1).requires_grad_() for _ in range(2))
    leaves = (a, b) if op in ("mul", "div") else (a,)
    y = f(a, b)
    assert op == "logsumexp" or "Node" in y.grad_fn.name()
    dy = torch.randn_like(y)
    want = torch.autograd.grad(y, leaves, dy)
    def gradients(unpack):
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t.detach(), unpack):
            y = f(a, b)
        return torch.autograd.grad(y, leaves, dy)
    def strided(t):
        return torch.zeros(*t.shape, 2, device="cuda")[..., 0].copy_(t)
    assert all(torch.equal(p, q) for p, q in zip(gradients(strided), want))
    assert all(torch.equal(p, q) for p, q in zip(gradients(lambda t: strided(t.t()).t() if t.dim() == 2 else t), want))
    for unpack, error in ((lambda t: t.double(), TypeError), (lambda t: t.cpu(), RuntimeError), (lambda t: t[:0], ValueError)):
        with pytest.raises(error):
            gradients(unpack)
