"""The Python module of token steps' entry points (csrc/launch/launch.cpp): what it takes and refuses of a launch's tensors and numbers.
It looks at their shapes, types and places only, so CPU tensors do."""
import pytest
import torch

from loqa_hub_amd.ops import _lib

BF16, I32, F32 = torch.bfloat16, torch.int32, torch.float32


@pytest.fixture(scope="module")
def lib():
    return _lib.launch()


def _i32(*shape):
    return torch.zeros(*shape, dtype=I32)


def _odd(*shape, dtype):
    """Every second entry of the last dimension: not contiguous."""
    return torch.zeros(*shape[:-1], 2 * shape[-1], dtype=dtype)[..., ::2]


# ------------------------------------------------------------------ numbers, tensors and addresses
def test_arguments(lib):
    w, none = torch.zeros(4, dtype=BF16), [None, 0, 0, None, 0, 0, 0, 0, None, 0, 0, None]
    call = lib.loqa_head_product                      # no rows: returns at once
    assert call(*none) == 0 and call(w, True, -1, w.data_ptr(), 0, 1, 128, 64, w, 1 << 40, 0, 0) == 0
    for n in (0, 11, 13):
        with pytest.raises(TypeError, match="takes 12 arguments, got %d" % n):
            call(*(none + [0])[:n])
    for at, bad, error in ((0, "x", TypeError), (0, 1.5, TypeError), (3, [w], TypeError), (0, 1 << 64, OverflowError), (1, 1 << 63, OverflowError),
                           (1, 1.0, TypeError), (4, 1 << 31, OverflowError), (4, -(1 << 31) - 1, OverflowError), (5, None, TypeError),
                           (0, torch.zeros(2, 2).to_sparse(), RuntimeError)):
        with pytest.raises(error):
            call(*[bad if i == at else x for i, x in enumerate(none)])
    with pytest.raises(TypeError):                    # a float argument
        lib.loqa_gated_rmsnorm(None, None, None, 0, 0, "eps", None, 0, 0, 1, 1, 0, None)


def test_types_of_pairs(lib):
    assert lib.i32c(_i32(3), "a", _i32(2, 2), "b") is None and lib.f32c(torch.zeros(3), "a") is None and lib.i32c() is None
    for fn, good, bad in ((lib.i32c, _i32(3), (torch.zeros(3), torch.zeros(3, dtype=torch.int64), _odd(3, dtype=I32), None, 7)),
                          (lib.f32c, torch.zeros(3), (_i32(3), torch.zeros(3, dtype=BF16), _odd(3, dtype=F32), None))):
        for x in bad:
            with pytest.raises(TypeError, match="second"):
                fn(good, "first", x, "second")


# ------------------------------------------------------------------ qk_shapes
H, G, D, T = 4, 2, 16, 5
QK = ("u", "k", "v", "pos", "slots", "cos", "H", "G", "D", "Dv", "v_off", "dims")


def _qk(**other):
    a = dict(u=torch.zeros(T, (H + G) * D + G * D + 3, dtype=BF16), k=torch.zeros(3, 8, G * D, dtype=BF16), v=torch.zeros(3, 8, G * D, dtype=BF16),
             pos=_i32(T), slots=_i32(T), cos=torch.zeros(7, 4, 2), H=H, G=G, D=D, Dv=D, v_off=(H + G) * D, dims=8)
    a.update(other)
    return [a[x] for x in QK]


def test_qk_shapes(lib):
    W = (H + G) * D + G * D + 3
    assert lib.qk_shapes(*_qk()) == (T, W, 3, 8, 7)
    assert lib.qk_shapes(*_qk(dims=0, cos=None)) == (T, W, 3, 8, 0)
    assert lib.qk_shapes(*_qk(u=torch.zeros(T, W + 9, dtype=BF16)[:, 9:], v_off=-1, pos=_i32(T + 2), slots=_i32(T + 1))) == (T, W + 9, 3, 8, 7)
    assert lib.qk_shapes(*_qk(v=torch.zeros(3, 8, G * 8, dtype=BF16), Dv=8)) == (T, W, 3, 8, 7)
    assert lib.qk_shapes(*_qk(k=torch.zeros(3, 8, G * D, 1, dtype=BF16))) == (T, W, 3, 8, 7)


@pytest.mark.parametrize("other,error", [
    (dict(u=torch.zeros(T, 2, 96, dtype=BF16)), AssertionError), (dict(u=_odd(T, 144, dtype=BF16)), AssertionError),
    (dict(u=torch.zeros(T, (H + G) * D - 1, dtype=BF16)), AssertionError), (dict(u=torch.zeros(T, (H + G) * D + G * D - 1, dtype=BF16)), AssertionError),
    (dict(v_off=(H + G) * D - 1), AssertionError), (dict(v_off=(H + G) * D + 4), AssertionError), (dict(v_off=-1, Dv=8), AssertionError),
    (dict(dims=7), AssertionError), (dict(dims=18), AssertionError), (dict(dims=-2), AssertionError), (dict(cos=None), AssertionError),
    (dict(cos=torch.zeros(7, 5, 2)), AssertionError), (dict(cos=torch.zeros(8)), AssertionError), (dict(cos=torch.zeros(7, 4, 2, dtype=BF16)), TypeError),
    (dict(cos=_odd(7, 4, dtype=F32)), TypeError),
    (dict(k=torch.zeros(3, 8, G * D + 1, dtype=BF16)), AssertionError), (dict(k=torch.zeros(3, 8 * G * D, dtype=BF16)), AssertionError),
    (dict(k=torch.zeros(3, 8, G * D)), AssertionError), (dict(k=_odd(3, 8, G * D, dtype=BF16)), AssertionError),
    (dict(v=torch.zeros(3, 8, G * D)), AssertionError), (dict(v=torch.zeros(4, 8, G * D, dtype=BF16)), AssertionError),
    (dict(v=torch.zeros(3, 9, G * D, dtype=BF16)), AssertionError), (dict(v=torch.zeros(3, 8, G * D - 1, dtype=BF16)), AssertionError),
    (dict(v=torch.zeros(3, 8, G * D, 1, dtype=BF16)), AssertionError), (dict(v=_odd(3, 8, G * D, dtype=BF16)), AssertionError),
    (dict(pos=_i32(T - 1)), AssertionError), (dict(pos=torch.zeros(T, dtype=torch.int64)), TypeError), (dict(pos=_odd(T, dtype=I32)), TypeError),
    (dict(slots=_i32(T - 1)), AssertionError), (dict(slots=torch.zeros(T)), TypeError), (dict(slots=None), AssertionError), (dict(u=3), TypeError),
    (dict(H="x"), TypeError), (dict(H=1 << 63), OverflowError)])
def test_qk_shapes_refuses(lib, other, error):
    with pytest.raises(error):
        lib.qk_shapes(*_qk(**other))


# ------------------------------------------------------------------ window_shapes
WIN = ("q", "k", "v", "cu", "ctx", "bt", "pos", "H", "G", "D", "Dv")


def _win(H=H, G=G, D=D, Dv=None, dtype=BF16, **other):
    Dv = D if Dv is None else Dv
    a = dict(q=torch.zeros(T, H * D, dtype=dtype), k=torch.zeros(3, 8, G * D, dtype=dtype), v=torch.zeros(3, 8, G * Dv, dtype=dtype), cu=_i32(3), ctx=_i32(2),
             bt=_i32(2, 6), pos=_i32(T), H=H, G=G, D=D, Dv=Dv)
    a.update(other)
    return [a[x] for x in WIN]


def _off(*shape):
    return torch.zeros(4 + torch.Size(shape).numel(), dtype=BF16)[4:].view(*shape)


@pytest.mark.parametrize("kw,token", [({}, True), (dict(D=128), True), (dict(D=136), False), (dict(D=128, Dv=136), False), (dict(D=20), False), (dict(Dv=20), False),
                                      (dict(H=32), True), (dict(H=34), False), (dict(dtype=F32), False), (dict(q=_off(T, H * D)), False),
                                      (dict(k=_off(3, 8, G * D)), False), (dict(v=_off(3, 8, G * D)), False), (dict(D=512), False)])
def test_window_shapes(lib, kw, token):
    """The last says whether the matrix-core token form takes the rows, for which the caller then sizes a workspace."""
    assert lib.window_shapes(*_win(**kw)) == (T, 3, 8, 2, 6, token)


@pytest.mark.parametrize("other,error", [
    (dict(q=torch.zeros(T, H * D + 1, dtype=BF16)), AssertionError), (dict(q=torch.zeros(T, H * D)), AssertionError), (dict(q=torch.zeros(T, dtype=BF16)), AssertionError),
    (dict(q=torch.zeros(T, 2 * H * D, dtype=BF16)[:, ::2]), AssertionError), (dict(H=5), AssertionError), (dict(G=3), AssertionError),
    (dict(k=torch.zeros(3, 8, G * D)), AssertionError), (dict(k=torch.zeros(3, 8, G * D + 8, dtype=BF16)), AssertionError), (dict(k=_odd(3, 8, G * D, dtype=BF16)), AssertionError),
    (dict(v=torch.zeros(2, 8, G * D, dtype=BF16)), AssertionError), (dict(v=torch.zeros(3, 4, G * D, dtype=BF16)), AssertionError), (dict(v=None), AssertionError),
    (dict(D=520), AssertionError), (dict(Dv=520), AssertionError),
    (dict(cu=_i32(2)), AssertionError), (dict(cu=_i32(4)), AssertionError), (dict(cu=torch.zeros(3)), TypeError), (dict(ctx=_i32(3)), AssertionError),
    (dict(ctx=torch.zeros(2, dtype=torch.int64)), TypeError), (dict(bt=_i32(12)), AssertionError), (dict(bt=_i32(1, 6)), AssertionError),
    (dict(bt=_odd(2, 6, dtype=I32)), TypeError), (dict(pos=_i32(T - 1)), AssertionError), (dict(pos=torch.zeros(T)), TypeError), (dict(pos="x"), TypeError)])
def test_window_shapes_refuses(lib, other, error):
    with pytest.raises(error):
        lib.window_shapes(*_win(**other))


def test_shapes_count_their_arguments(lib):
    for fn, args in ((lib.qk_shapes, _qk()), (lib.window_shapes, _win())):
        for bad in (args[:-1], args + [0]):
            with pytest.raises(TypeError, match="arguments"):
                fn(*bad)
    with pytest.raises(AssertionError):               # no division by no key heads
        lib.window_shapes(*_win()[:8], 0, D, D)
