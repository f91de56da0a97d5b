"""The entry points' native call path against the Python path: every form it
takes gives the same bits as the same call with caller-supplied buffers (which
it leaves to the Python code), and it declines everything else."""

from pathlib import Path
import subprocess
import sys

import pytest
import torch

from mini_engine_hip import build
from mini_engine_hip.kernels import hip_extension as ext
from mini_engine_hip.kernels.data import write_kv_cache_slots
from mini_engine_hip.kernels.linear import linear_rows
from mini_engine_hip.kernels.paged import paged_attention, paged_attention_decode_write
from mini_engine_hip.kernels.prefill import paged_prefill_attention, prefill_attention
from mini_engine_hip.kernels.rope import qk_norm_rope_write_kv

DEV = "cuda"


class Subclass(torch.Tensor):
    pass


def decode_args(device, dtype=torch.bfloat16, batch=3, heads=4, kv=2, dim=64, block=16, width=9):
    gen = torch.Generator().manual_seed(7)
    key, value = (torch.randn(batch * width + 2, block, kv, dim, generator=gen).to(dtype) for _ in range(2))
    table = torch.randperm(batch * width + 2, generator=gen)[:batch * width].view(batch, width)
    lens = torch.tensor([1 + 40 * i for i in range(batch)])
    q = torch.randn(batch, heads, dim, generator=gen).to(dtype)
    return [t.to(device) for t in (q, key, value, table, lens)] + [block]


def test_declines_what_is_not_plain():
    """CPU tensors, subclasses, wrong argument types: None, and no error."""
    native = ext.native_calls()
    args = decode_args("cpu")
    assert native.decode(*args, 0) is None
    assert native.decode(*args[:5], 16.0, 0) is None
    assert native.decode(args[0].as_subclass(Subclass), *args[1:], 0) is None
    assert native.decode(None, *args[1:], 0) is None
    assert native.decode() is None
    q, k, v = (torch.zeros(1, 2, 4, 64) for _ in range(3))
    assert native.dense(q, k, v, 0) is None
    assert native.linear(torch.zeros(2, 64), torch.zeros(32, 64), None) is None
    with pytest.raises(RuntimeError, match="must be CUDA"):
        paged_attention(*args, validate=False)


def test_bind_refuses_a_wrong_library():
    with pytest.raises(ValueError):
        ext.native_calls().bind(len, (1, 2))


REFUSED = """
import torch
from mini_engine_hip import HipLinear, build, linear_rows, paged_attention, paged_prefill_attention, prefill_attention
from mini_engine_hip import qk_norm_rope_write_kv, write_kv_cache_slots
from mini_engine_hip.kernels.paged import paged_attention_decode_write

def no_build(**_):
    raise SystemExit("a refused call went to the library")

build.library_path = lambda: build.PACKAGE_DIR / "absent.so"
build.build_library = no_build
half, i64 = lambda *s: torch.zeros(*s).half(), lambda *s: torch.zeros(*s, dtype=torch.int64)
cache, rows, row = half(2, 16, 2, 64), half(1, 4, 64), half(1, 2, 64)
calls = [
    (ValueError, lambda: HipLinear(64, 32)(torch.zeros(2, 64))),
    (ValueError, lambda: linear_rows(half(2, 64), half(32, 64))),
    (ValueError, lambda: prefill_attention(half(1, 4, 3, 64), half(1, 2, 3, 64), half(1, 2, 3, 64))),
    (ValueError, lambda: paged_prefill_attention(rows, cache, cache, i64(2), i64(1), i64(1, 2), i64(1), 16, validate=False)),
    (RuntimeError, lambda: paged_attention(rows, cache, cache, i64(1, 2), i64(1), 16, validate=False)),
    (RuntimeError, lambda: paged_attention_decode_write(rows, cache, cache, i64(1, 2), i64(1), 16, row, row, validate=False)),
    (ValueError, lambda: write_kv_cache_slots(cache, cache, i64(1), row, row, validate=False)),
    (RuntimeError, lambda: qk_norm_rope_write_kv(rows, row, row, half(64), half(64), half(1, 32), half(1, 32), cache, cache,
                                                 slot_mapping=i64(1), validate=False)),
]
for kind, call in calls:
    try:
        call()
    except kind as error:
        assert "library" not in str(error), error
    else:
        raise SystemExit("not refused")
"""


def test_refused_calls_need_no_library():
    """What the entry points refuse is refused before any library is looked for."""
    done = subprocess.run([sys.executable, "-c", REFUSED], cwd=build.PACKAGE_DIR.parent, capture_output=True, text=True, timeout=300)
    assert done.returncode == 0, done.stderr[-2000:]


@pytest.fixture
def fresh_loader(monkeypatch):
    """The loader as in a new process; the process's own state comes back afterwards."""
    monkeypatch.setattr(ext, "native", ext.NoNativeCalls())
    caches = (ext.load_hip_extension, ext._host_module)
    for cached in caches:
        cached.cache_clear()
    yield monkeypatch
    for cached in caches:
        cached.cache_clear()


@pytest.mark.parametrize("content", [None, b"no shared object"])
def test_python_path_serves_without_the_native_one(fresh_loader, tmp_path, content):
    """A host module that is missing or cannot be loaded: a warning, and every
    call is left to the Python code."""
    planted = tmp_path / "mvme_host.so"
    if content is not None:
        planted.write_bytes(content)
    fresh_loader.setattr(build, "host_path", lambda: planted)
    with pytest.warns(RuntimeWarning, match="Python path"):
        lib = ext.load_hip_extension()
    assert lib.workspace_size(4, 16, 8, 128, 16, 64, 64) > 0
    assert ext.native.decode(*decode_args("cpu"), 0) is None


@pytest.mark.parametrize("name,value", [("__version__", "0.0"), ("version.git_version", "f" * 40)])
def test_another_torch_needs_another_native_path(fresh_loader, name, value):
    """The module inlines torch's headers: one built for another torch is not loaded."""
    fresh_loader.setattr(f"torch.{name}", value)
    with pytest.warns(RuntimeWarning, match="another torch"):
        ext.load_hip_extension()
    assert isinstance(ext.native, ext.NoNativeCalls)


def test_native_path_without_a_digest_is_left_out(fresh_loader, tmp_path):
    fresh_loader.setattr(build, "host_digest_path", lambda: tmp_path / "absent")
    with pytest.warns(RuntimeWarning, match="no build digest"):
        ext.load_hip_extension()
    assert isinstance(ext.native, ext.NoNativeCalls)


def test_library_is_built_where_the_native_path_cannot_be(fresh_loader, tmp_path):
    """No host compiler or torch headers: the library needs neither."""
    built = build.library_path()
    fresh_loader.setattr(build, "LIB_DIR", tmp_path)
    fresh_loader.setattr(build, "PACKAGE_DIR", tmp_path)

    def run(cmd):
        if "host_calls.cpp" in " ".join(cmd):
            raise RuntimeError("no host compiler")
        target = Path(cmd[cmd.index("-o") + 1])
        target.write_bytes(built.read_bytes() if ".so" in target.name else b"")

    fresh_loader.setattr(build, "_run", run)
    with pytest.warns(RuntimeWarning, match="Python path"):
        lib = ext.load_hip_extension()
    assert lib.path == tmp_path / build.LIB_NAME
    with pytest.raises(RuntimeError, match="no host compiler"):
        build.build_library()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("dim", [64, 80, 128])
@pytest.mark.parametrize("partition", [0, 64, -1])
def test_decode_equals_the_python_path(dtype, dim, partition):
    args = decode_args(DEV, dtype, dim=dim)
    assert ext.native_calls().decode(*args, partition) is not None
    out = torch.empty_like(args[0])
    paged_attention(*args, validate=False, partition_tokens=partition, out=out)
    assert torch.equal(paged_attention(*args, validate=False, partition_tokens=partition), out)


@pytest.mark.gpu
@pytest.mark.parametrize("rope", [False, True])
@pytest.mark.parametrize("layout", ["split", "dense", "misaligned"])
def test_decode_write_equals_the_python_path(rope, layout):
    dtype, heads, kv, dim = torch.bfloat16, 4, 2, 64
    base, key, value, table, lens, block = decode_args(DEV, dtype)
    gen = torch.Generator().manual_seed(3)
    qkv = torch.randn(3, heads + 2 * kv, dim, generator=gen).to(dtype).to(DEV)
    q, nk, nv = qkv.split([heads, kv, kv], dim=1)
    if layout != "split" or not rope:
        q = q.contiguous()
    if layout != "split":
        nk, nv = nk.contiguous(), nv.contiguous()
    if layout == "misaligned":  # 2-byte offset: the two launches of the Python path
        nk = torch.cat([nk.flatten()[:1], nk.flatten()])[1:].view(nk.shape)
        assert nk.data_ptr() % 16 != 0
    cos, sin = torch.rand(3, dim // 2, generator=gen).to(dtype).to(DEV), torch.rand(3, dim // 2, generator=gen).to(dtype).to(DEV)
    weight = torch.rand(dim, generator=gen).to(dtype).to(DEV)
    extra = dict(q_weight=weight, k_weight=weight, cos=cos, sin=sin) if rope else {}
    k1, v1, k2, v2 = key.clone(), value.clone(), key.clone(), value.clone()
    out = torch.empty(3, heads, dim, dtype=dtype, device=DEV)
    paged_attention_decode_write(q, k1, v1, table, lens, block, nk, nv, validate=False, out=out, **extra)
    got = paged_attention_decode_write(q, k2, v2, table, lens, block, nk, nv, validate=False, **extra)
    assert torch.equal(got, out) and torch.equal(k1, k2) and torch.equal(v1, v2)
    values = [extra.get(n) for n in ("q_weight", "k_weight", "cos", "sin")]
    taken = ext.native_calls().decode_write(q, k2, v2, table, lens, block, nk, nv, *values, 1e-6, 0) is not None
    assert taken == (layout != "misaligned")


@pytest.mark.gpu
@pytest.mark.parametrize("new", [[5, 40], [300, 1]])
def test_prefill_write_and_rope_equal_the_python_path(new):
    dtype, heads, kv, dim, block = torch.float16, 4, 2, 128, 16
    gen = torch.Generator().manual_seed(new[0])
    tokens, starts = sum(new), torch.tensor([100, 0])
    lens = starts + torch.tensor(new)
    width = -(-int(lens.max()) // block)
    key, value = (torch.randn(2 * width, block, kv, dim, generator=gen).to(dtype).to(DEV) for _ in range(2))
    table = torch.randperm(2 * width, generator=gen).view(2, width)
    slots = torch.cat([table[i, p // block] * block + p % block
                       for i in range(2) for p in [torch.arange(starts[i], lens[i])]]).to(DEV)
    cu = torch.tensor([0, new[0], tokens]).to(DEV)
    table, starts, lens = table.to(DEV), starts.to(DEV), lens.to(DEV)
    q, k, v = torch.randn(tokens, heads + 2 * kv, dim, generator=gen).to(dtype).to(DEV).split([heads, kv, kv], dim=1)
    cos, sin = torch.rand(2, tokens, dim // 2, generator=gen).to(dtype).to(DEV)
    weight = torch.rand(dim, generator=gen).to(dtype).to(DEV)
    caches = [[key.clone(), value.clone()] for _ in range(2)]
    out = torch.empty(tokens, heads, dim, dtype=dtype, device=DEV)
    rope = lambda c, **kw: qk_norm_rope_write_kv(q, k, v, weight, weight, cos, sin, *c, slot_mapping=slots,  # noqa: E731
                                                 validate=False, **kw)
    assert torch.equal(rope(caches[0]), rope(caches[1], out=out))
    assert all(torch.equal(a, b) and not torch.equal(a, c) for a, b, c in zip(*caches, (key, value)))
    native = ext.native_calls()
    again = [key.clone(), value.clone()]
    assert native.rope_slots(q, k, v, weight, weight, cos, sin, *again, slots, 1e-6) is not None
    assert all(torch.equal(a, b) for a, b in zip(again, caches[1]))
    rows = torch.randn(2, tokens, kv, dim, generator=gen).to(dtype).to(DEV)
    write_kv_cache_slots(*caches[0], slots, *rows, validate=False)
    write_kv_cache_slots(*caches[1], slots, *rows)
    assert all(torch.equal(a, b) and not torch.equal(a, c) for a, b, c in zip(*caches, again))
    assert native.write_slots(*again, slots, *rows) is True
    assert all(torch.equal(a, b) for a, b in zip(again, caches[1]))
    args = (out, *caches[0], cu, starts, table, lens, block)
    assert native.prefill(*args, 0) is not None
    workspace = torch.empty(1 << 24, dtype=torch.uint8, device=DEV)
    assert torch.equal(paged_prefill_attention(*args, validate=False),
                       paged_prefill_attention(*args, validate=False, workspace=workspace))


@pytest.mark.gpu
@pytest.mark.parametrize("dim,view", [(128, True), (128, False), (64, True), (100, False)])
def test_dense_and_linear_equal_the_python_path(dim, view):
    gen = torch.Generator().manual_seed(dim)
    make = lambda n, h: (torch.randn(n, h, dim, generator=gen).bfloat16().to(DEV).transpose(0, 1).unsqueeze(0))  # noqa: E731
    q, k, v = make(70, 4), make(90, 2), make(90, 2)
    if not view:
        q, k, v = q.contiguous(), k.contiguous(), v.contiguous()
    out = torch.empty(1, 4, 70, dim, dtype=q.dtype, device=DEV)
    result = prefill_attention(q, k, v, query_start=20)
    assert torch.equal(result, prefill_attention(q, k, v, query_start=20, out=out))
    assert result.stride() == (70 * 4 * dim, dim, 4 * dim, 1)
    assert (ext.native_calls().dense(q, k, v, 20) is not None) == (dim % 8 == 0)
    x, weight = torch.randn(7, 512, generator=gen).bfloat16().to(DEV), torch.randn(64, 512, generator=gen).bfloat16().to(DEV)
    bias = torch.randn(64, generator=gen).bfloat16().to(DEV)
    for b in (None, bias):
        buffer = torch.empty(7, 64, dtype=x.dtype, device=DEV)
        assert torch.equal(linear_rows(x, weight, b), linear_rows(x, weight, b, out=buffer))
        assert ext.native_calls().linear(x, weight, b) is not None
    assert torch.equal(linear_rows(x[:, ::1][:3], weight), linear_rows(x, weight)[:3])


@pytest.mark.gpu
def test_declines_layouts_of_the_python_path():
    """Layouts that the kernels cannot read in place, and types they do not take, are
    left to the Python code: misaligned and oddly strided rows, FP32, other devices'
    and other types' metadata."""
    native = ext.native_calls()
    flat = torch.randn(1 + 70 * 4 * 64, device=DEV).bfloat16()
    plain, shifted = (flat[i:i + 70 * 4 * 64].view(1, 4, 70, 64) for i in (0, 1))
    assert native.dense(plain, plain, plain, 0) is not None
    for q, k, v in ((shifted, plain, plain), (plain, shifted, shifted), (plain, plain, plain.transpose(1, 2).contiguous().transpose(1, 2)),
                    (plain[..., ::2], plain[..., ::2], plain[..., ::2]), (plain.float(),) * 3):
        assert native.dense(q, k, v, 0) is None
    assert native.dense(plain, plain, plain, True) is None and native.dense(plain, plain, plain, 1) is None
    x, weight = torch.randn(4, 68, device=DEV).bfloat16()[:, :64], torch.randn(32, 64, device=DEV).bfloat16()
    assert native.linear(x.contiguous(), weight, None) is not None
    for a, w, b in ((x, weight, None), (x.contiguous().float(), weight.float(), None), (x.contiguous(), weight.t().contiguous().t(), None),
                    (x.contiguous(), weight, torch.zeros(31, device=DEV).bfloat16()), (x.contiguous()[None], weight, None)):
        assert native.linear(a, w, b) is None
    q, key, value, table, lens, block = decode_args(DEV)
    rows = torch.randn(3, 2, 64, device=DEV).bfloat16()
    slots = torch.tensor([3, 20, 40], device=DEV)
    assert native.write_slots(key, value, slots, rows, rows) is True
    for args in ((key, value, slots.int(), rows, rows), (key, value, slots.cpu(), rows, rows), (key.float(), value.float(), slots, rows.float(), rows.float()),
                 (key, value, slots, rows.transpose(1, 2).contiguous().transpose(1, 2), rows), (key, value, slots[:2], rows, rows)):
        assert native.write_slots(*args) is None
    weight, trig = torch.rand(64, device=DEV).bfloat16(), torch.rand(3, 32, device=DEV).bfloat16()
    rope = (q, rows, rows, weight, weight, trig, trig, key, value, slots)
    assert native.rope_slots(*rope, 1e-6) is not None
    assert native.rope_slots(*rope, 0.0) is None and native.rope_slots(*rope, 1) is None
    assert native.rope_slots(*rope[:5], trig.float(), trig.float(), *rope[7:], 1e-6) is None
    cu, starts = torch.tensor([0, 1, 2, 3], device=DEV), lens - 1
    assert native.prefill(q, key, value, cu, starts, table, lens, block, 0) is not None
    for args in ((q.float(), key.float(), value.float(), cu, starts, table, lens), (q, key, value, cu.int(), starts, table, lens),
                 (q, key, value, cu, starts, table.t().contiguous().t(), lens), (q[:, :, ::2], key, value, cu, starts, table, lens)):
        assert native.prefill(*args, block, 0) is None
