"""The C-ABI boundary, without a GPU: the built library loads, exports every entry point that
include/*.h declares, the ctypes bindings agree with the header's parameter lists, and the
host-side contract checks (status codes, workspace sizing) behave as documented.  Nothing here
launches a kernel."""
import glob
import os
import re
import subprocess
import sys

import pytest
import torch

from pto_fuser_amd import _build, _hip

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _header_functions():
    """name -> parameter count, for every function prototype in include/*.h."""
    out = {}
    for h in glob.glob(os.path.join(ROOT, "include", "*.h")):
        text = re.sub(r"/\*.*?\*/", " ", open(h).read(), flags=re.S)
        text = re.sub(r"//[^\n]*", " ", text)
        for m in re.finditer(r"\b(pf_\w+)\s*\(([^;{)]*)\)\s*;", text):
            params = [p for p in m.group(2).split(",") if p.strip() and p.strip() != "void"]
            out[m.group(1)] = len(params)
    return out


@pytest.fixture(scope="module")
def lib():
    _build.ensure_built()
    return _hip.load()


def test_header_declares_entry_points():
    fns = _header_functions()
    for name in ("pf_gdn_exec", "pf_gdn_setup", "pf_gdn_teardown", "pf_tri_inv_exec",
                 "pf_kkt_inv_exec", "pf_gdn_chunk_local_exec", "pf_gdn_scan_output_exec"):
        assert name in fns, name


def test_library_exports_every_declared_symbol(lib):
    fns = _header_functions()
    missing = [n for n in fns if not hasattr(lib, n)]
    assert not missing, f"declared but not exported: {missing}"


def test_bindings_match_header_arity(lib):
    fns = _header_functions()
    assert set(_hip.SIGNATURES) == set(fns), (set(_hip.SIGNATURES) ^ set(fns))
    for name, (_, argtypes) in _hip.SIGNATURES.items():
        assert len(argtypes) == fns[name], f"{name}: binding has {len(argtypes)} args, header {fns[name]}"


def test_status_strings_and_version(lib):
    assert lib.pf_abi_version() >= 1
    assert _hip.status_text(_hip.PF_OK) == "ok"
    assert "argument" in _hip.status_text(_hip.PF_ERR_ARG)
    assert "workspace" in _hip.status_text(_hip.PF_ERR_WORKSPACE)


def test_workspace_sizing_contract(lib):
    # bf16: T (bf16) + G (fp32), each 256-byte aligned, + a 256-byte slot for the scale (the
    # bf16 scan forms P itself); fp32: T + P (fp32) + G + the slot
    M = 4 * 16 * 64
    al = lambda n: (n + 255) // 256 * 256
    want = al(M * 64 * 64 * 2) + al(M * 64 * 4) + 256
    assert lib.pf_gdn_workspace_bytes(4, 16, 4096, 64, 128, 128, _hip.PF_DTYPE_BF16) == want
    want32 = 2 * al(M * 64 * 64 * 4) + al(M * 64 * 4) + 256
    assert lib.pf_gdn_workspace_bytes(4, 16, 4096, 64, 128, 128, _hip.PF_DTYPE_F32) == want32
    # unsupported shapes / dtypes report size 0 and setup refuses them
    assert lib.pf_gdn_workspace_bytes(1, 1, 100, 64, 128, 128, 1) == 0      # T % C != 0
    assert lib.pf_gdn_workspace_bytes(1, 1, 128, 32, 128, 128, 1) == 0      # C != 64
    assert lib.pf_gdn_workspace_bytes(1, 1, 128, 64, 64, 128, 1) == 0       # DK != 128
    assert lib.pf_gdn_workspace_bytes(1, 1, 128, 64, 128, 128, 7) == 0      # bad dtype
    # the longest chain: 2^22 tokens (32-bit per-chain addressing); one chunk more is refused
    assert lib.pf_gdn_workspace_bytes(1, 1, 1 << 22, 64, 128, 128, 1) > 0
    assert lib.pf_gdn_workspace_bytes(1, 1, (1 << 22) + 64, 64, 128, 128, 1) == 0
    assert lib.pf_gdn_exec(None, None, None, None, None, None, None, None, 1, 1, (1 << 22) + 64, 64,
                           128, 128, 1, 0.1, None, None) == _hip.PF_ERR_ARG
    assert not lib.pf_gdn_setup(1, 1, 100, 64, 128, 128, 1)


def test_gdn_workspace_of_segmented_chains():
    """Few long chains ask for the segments' maps and states (two 128 x 128 fp32 matrices each) on top of
    what whole chains need, and the fp32 size of a shape always covers its bf16 one."""
    lib = _hip.load()

    def size(B, H, T, dt):
        return lib.pf_gdn_workspace_bytes(B, H, T, 64, 128, 128, dt)

    base = (1 << 15) // 64 * 4 * (64 * 64 * 2 + 64 * 4) + 256
    extra = size(1, 4, 1 << 15, _hip.PF_DTYPE_BF16) - base
    assert extra > 0 and extra % (4 * 2 * 128 * 128 * 4) == 0
    for B, H, T in ((1, 1, 64), (1, 1, 1024), (1, 4, 1 << 15), (1, 8, 4096), (2, 5, 5120), (4, 16, 4096),
                    (1, 1, 1 << 22), (1, 32, 1 << 15)):
        assert size(B, H, T, _hip.PF_DTYPE_F32) >= size(B, H, T, _hip.PF_DTYPE_BF16) > 0


def test_workspace_sizes_start_no_runtime(lib):
    """Sizes are arithmetic: a process that only asks for them (before it forks, say) does not start the HIP
    runtime.  Every HIP call is logged at this level; the last one is there to show that."""
    code = ("import ctypes, sys\n"
            "lib = ctypes.CDLL(sys.argv[1])\n"
            "for f in (lib.pf_gdn_workspace_bytes, lib.pf_kda_workspace_bytes):\n"
            "    f.restype, f.argtypes = ctypes.c_size_t, [ctypes.c_int] * 7\n"
            "    assert f(1, 4, 32768, 64, 128, 128, 0) >= f(1, 4, 32768, 64, 128, 128, 1) > 0\n"
            "print('sized', file=sys.stderr, flush=True)\n"
            "lib.hipGetDeviceCount(ctypes.byref(ctypes.c_int()))\n")
    run = subprocess.run([sys.executable, "-c", code, _hip.lib_path()], capture_output=True, text=True,
                         env={**os.environ, "AMD_LOG_LEVEL": "3"}, timeout=120)
    assert run.returncode == 0, run.stderr[-2000:]
    before, after = run.stderr.split("sized", 1)
    assert "hipGetDevice" in after and "hip" not in before, before[-2000:]


def _segments(lib, op, chains, chunks):
    """Segments per chain that the workspace of a bf16 shape holds (1: whole chains)."""
    size = lib.pf_gdn_workspace_bytes if op == "gdn" else lib.pf_kda_workspace_bytes
    extra = size(1, chains, 64 * chunks, 64, 128, 128, 1) - size(1, chains * chunks, 64, 64, 128, 128, 1)
    assert extra % (chains * 2 * 128 * 128 * 4) == 0
    return 1 + extra // (chains * 2 * 128 * 128 * 4)


@pytest.mark.parametrize("op,chains,chunks,segmented", [
    ("gdn", 1, 128, True), ("gdn", 4, 512, True), ("gdn", 8, 64, True), ("gdn", 8, 256, True),
    ("gdn", 16, 128, True), ("gdn", 32, 512, True), ("gdn", 1, 32, True), ("gdn", 20, 96, True),
    ("gdn", 12, 40, False), ("gdn", 33, 192, False), ("gdn", 64, 256, False), ("gdn", 15, 23, False),
    ("kda", 1, 128, True), ("kda", 4, 128, True), ("kda", 8, 64, True), ("kda", 16, 128, True),
    ("kda", 24, 128, True), ("kda", 32, 256, True),
    ("kda", 9, 24, False), ("kda", 8, 28, False), ("kda", 16, 32, False), ("kda", 32, 64, False)])
def test_chains_run_in_segments_where_that_was_faster(lib, op, chains, chunks, segmented):
    """The rule's decisions at shapes measured both ways (the times are beside the rule)."""
    assert (_segments(lib, op, chains, chunks) > 1) == segmented


def test_segment_states_are_bounded(lib):
    """The segments' states and maps never take more than 32 MiB (GDN) or 16 MiB (KDA) beside what whole
    chains need: their maps run in one generation of workgroups."""
    for op, mib in (("gdn", 32), ("kda", 16)):
        for chains in (1, 3, 8, 16, 17, 36, 64, 100, 132, 256, 300):
            for chunks in (16, 67, 128, 500, 512, 5040, 50000):
                assert (_segments(lib, op, chains, chunks) - 1) * chains * 2 * 128 * 128 * 4 <= mib << 20


@pytest.mark.parametrize("op", ["gdn", "kda"])
def test_chain_counts_do_not_wrap(lib, op):
    """B * H past 32 bits is refused: it may not come out as a small workspace that a call would accept."""
    size = lib.pf_gdn_workspace_bytes if op == "gdn" else lib.pf_kda_workspace_bytes
    for B, H in ((1 << 16, 1 << 16), ((1 << 16) + 1, (1 << 16) + 1), (1 << 20, 1 << 12), (1 << 15, 1 << 16)):
        assert size(B, H, 64, 64, 128, 128, 1) == 0
        assert size(B, H, 64, 64, 128, 128, 0) == 0
    assert size(1 << 12, 1 << 12, 64, 64, 128, 128, 1) >= (1 << 24) * 64 * 64 * 2


_FAKE_HIP = """#include <stdlib.h>
int mallocs, frees;
int hipMalloc(void** p, size_t n) { ++mallocs; *p = malloc(1); return 0; }
int hipFree(void* p) { ++frees; free(p); return 0; }
int hipDeviceSynchronize(void) { return 0; }
"""


@pytest.mark.parametrize("op", ["gdn", "kda"])
def test_a_shape_of_fewer_chunks_never_grows_a_handle(lib, tmp_path, op):
    """After a reserve for the most chunks a caller uses, a reserve for fewer allocates and frees nothing, also
    where those chains would run in segments and a fresh handle of theirs is larger: a graph captured
    on the handle keeps its buffer.  The library's allocations are counted in a process of its own."""
    src, so = tmp_path / "fake.c", tmp_path / "fake.so"
    src.write_text(_FAKE_HIP)
    subprocess.run(["gcc", "-shared", "-fPIC", str(src), "-o", str(so)], check=True)
    code = f"""
import ctypes, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
lib = ctypes.CDLL(sys.argv[2])
size, reserve, create = lib.pf_{op}_workspace_bytes, lib.pf_{op}_reserve, lib.pf_{op}_create
size.restype, size.argtypes = ctypes.c_size_t, [ctypes.c_int] * 7
reserve.argtypes, create.restype = [ctypes.c_void_p] + [ctypes.c_int] * 7, ctypes.c_void_p
count = lambda: (ctypes.c_int.in_dll(fake, "mallocs").value, ctypes.c_int.in_dll(fake, "frees").value)
ws = create()
large, small = (1, 64, 64 * 32, 64, 128, 128, 1), (1, 4, 64 * 500, 64, 128, 128, 1)
assert size(*small) > size(*large), "the shape of fewer chunks is the larger workspace"
assert reserve(ws, *large) == 0 and count() == (1, 0), count()
assert reserve(ws, *small) == 0 and count() == (1, 0), count()
assert reserve(ws, 1, 64, 64 * 64, 64, 128, 128, 1) == 0 and count() == (2, 1), count()
"""
    run = subprocess.run([sys.executable, "-c", code, str(so), _hip.lib_path()], capture_output=True, text=True,
                         timeout=120)
    assert run.returncode == 0, run.stderr[-2000:]


@pytest.mark.parametrize("B,H,T,C", [(1, 1, 64, 64), (4, 16, 4096, 64), (1, 32, 32768, 128),
                                     (3, 5, 192, 64)])
def test_fp32_workspace_holds_bf16(lib, B, H, T, C):
    """A handle reserved for the fp32 layout of a shape serves the bf16 call of that shape
    without growing (the integration stub reserves it so)."""
    for fn in (lib.pf_gdn_workspace_bytes, lib.pf_kda_workspace_bytes):
        f32 = fn(B, H, T, C, 128, 128, _hip.PF_DTYPE_F32)
        b16 = fn(B, H, T, C, 128, 128, _hip.PF_DTYPE_BF16)
        assert 0 < b16 <= f32


def test_kda_workspace_and_rejects(lib):
    # W, QE, k e^-G (bf16 [M,C,128] each) + T diag(beta) (bf16 [M,C,C]) + DEC (fp32 [M,128]),
    # 256-B aligned
    M = 2 * 32 * 128
    want = 3 * ((M * 64 * 128 * 2 + 255) // 256 * 256) + (M * 64 * 64 * 2 + 255) // 256 * 256 \
        + (M * 128 * 4 + 255) // 256 * 256
    assert lib.pf_kda_workspace_bytes(2, 32, 8192, 64, 128, 128, _hip.PF_DTYPE_BF16) == want
    # fp32 operands: W, U, QE, KR, P and DEC in fp32
    M1 = 128
    want32 = 4 * ((M1 * 64 * 128 * 4 + 255) // 256 * 256) + (M1 * 64 * 64 * 4 + 255) // 256 * 256 \
        + (M1 * 128 * 4 + 255) // 256 * 256
    assert lib.pf_kda_workspace_bytes(1, 1, 8192, 64, 128, 128, _hip.PF_DTYPE_F32) == want32
    assert lib.pf_kda_workspace_bytes(1, 1, 64, 64, 128, 128, _hip.PF_DTYPE_F32) > 0     # one chunk
    assert lib.pf_kda_workspace_bytes(1, 1, 64, 64, 128, 128, _hip.PF_DTYPE_BF16) > 0    # bf16 too
    assert lib.pf_kda_workspace_bytes(1, 1, 96, 64, 128, 128, _hip.PF_DTYPE_BF16) == 0   # T % C
    assert not lib.pf_kda_setup(1, 1, 100, 64, 128, 128, 1)
    assert lib.pf_kda_workspace_bytes(1, 1, 1 << 22, 64, 128, 128, 1) > 0
    assert lib.pf_kda_workspace_bytes(1, 1, (1 << 22) + 64, 64, 128, 128, 1) == 0
    assert lib.pf_kda_exec(None, None, None, None, None, None, None, None, 1, 1, 128, 64, 128, 128,
                           1, 0.1, None, None) == _hip.PF_ERR_WORKSPACE
    assert lib.pf_kda_exec(None, None, None, None, None, None, None, None, 1, 1, 128, 64, 128, 128,
                           0, 0.1, None, None) == _hip.PF_ERR_WORKSPACE                  # fp32 shape ok
    assert lib.pf_kda_exec(None, None, None, None, None, None, None, None, 1, 1, 128, 64, 128, 128,
                           7, 0.1, None, None) == _hip.PF_ERR_ARG                        # no such dtype
    assert lib.pf_kda_exec(None, None, None, None, None, None, None, None, 1, 1, 64, 64, 128, 128,
                           1, 0.1, None, None) == _hip.PF_ERR_WORKSPACE                  # bf16, one chunk
    assert lib.pf_kda_exec(None, None, None, None, None, None, None, None, 1, 1, 64, 64, 128, 64,
                           1, 0.1, None, None) == _hip.PF_ERR_ARG                        # dv 64


def test_exec_rejects_contract_violations_before_launch(lib):
    """Bad shapes, null pointers and missing workspaces return negative codes; nothing is
    enqueued (the calls are safe without a device)."""
    st = lib.pf_gdn_exec(None, None, None, None, None, None, None, None,
                         1, 1, 128, 64, 128, 128, 1, 0.1, None, None)
    assert st == _hip.PF_ERR_WORKSPACE
    st = lib.pf_gdn_exec(None, None, None, None, None, None, None, None,
                         1, 1, 100, 64, 128, 128, 1, 0.1, None, None)
    assert st == _hip.PF_ERR_ARG
    assert lib.pf_tri_inv_exec(None, None, 4, 64, None) == _hip.PF_ERR_ARG
    assert lib.pf_tri_inv_exec(1, 1, 4, 96, None) == _hip.PF_ERR_ARG       # unsupported C
    assert lib.pf_kkt_inv_exec(None, None, None, None, None, 4, 64, 128, 1, 0, None) == _hip.PF_ERR_ARG
    assert lib.pf_gdn_chunk_local_exec(None, None, None, None, 1, 1, 128, 64, 128, 128, 1,
                                       0.1, None, None) == _hip.PF_ERR_WORKSPACE
    assert lib.pf_gdn_scan_output_exec(None, None, None, None, None, None, None, 1, 1, 128, 64,
                                       128, 128, 1, None, None) == _hip.PF_ERR_WORKSPACE
    # stage kernels: null operands, unsupported (C, D, dtype) and bad output dtypes
    assert lib.pf_gated_qk_exec(None, None, None, None, None, None, None, None, 1, 1, 64, 128,
                                1, 1, 0, None) == _hip.PF_ERR_ARG
    assert lib.pf_gated_qk_exec(1, 1, None, None, None, None, None, 1, 1, 1, 16, 128,
                                1, 1, 0, None) == _hip.PF_ERR_ARG      # bf16 needs C >= 32
    assert lib.pf_gated_qk_exec(1, 1, None, None, None, None, None, 1, 1, 1, 64, 96,
                                0, 1, 0, None) == _hip.PF_ERR_ARG      # D = 96
    assert lib.pf_gated_qk_exec(1, 1, None, None, None, None, None, 1, 1, 1, 64, 128,
                                0, 1, 5, None) == _hip.PF_ERR_ARG      # out dtype
    assert lib.pf_qkv_flash_exec(1, 1, None, None, None, None, None, 1, 4, 64, 128, 1,
                                 None) == _hip.PF_ERR_ARG              # v missing
    assert lib.pf_qkv_flash_exec(1, 1, 1, None, None, None, None, 1, 4, 256, 128, 0,
                                 None) == _hip.PF_ERR_ARG              # C = 256
    assert lib.pf_scan_exec(1, 1, 1, None, None, 1, None, 1, 1, 2, 64, 128, 1, 0, 0,
                            None) == _hip.PF_ERR_ARG                   # decay missing
    assert lib.pf_scan_exec(1, 1, 1, 1, None, 1, None, 0, 1, 2, 64, 128, 1, 0, 0,
                            None) == _hip.PF_ERR_ARG                   # B = 0


def test_static_forward_rejects_on_host(lib):
    """The allocation-free forward refuses an input beyond its static scratch (8192 bf16 chunks)
    and unsupported shapes before touching the device (safe without one)."""
    st = lib.pf_gdn_exec_static(1, 1, 1, 1, 1, None, 1, None, 8, 16, 4096, 64, 128, 128,
                                _hip.PF_DTYPE_BF16, 0.1, None)
    assert st == _hip.PF_ERR_SCRATCH and "static scratch" in _hip.status_text(st)
    st = lib.pf_gdn_exec_static(1, 1, 1, 1, 1, None, 1, None, 1, 1, 100, 64, 128, 128,
                                _hip.PF_DTYPE_BF16, 0.1, None)
    assert st == _hip.PF_ERR_ARG                                         # T % C != 0
    st = lib.pf_gdn_exec_static(None, 1, 1, 1, 1, None, 1, None, 1, 1, 128, 64, 128, 128,
                                _hip.PF_DTYPE_BF16, 0.1, None)
    assert st == _hip.PF_ERR_ARG                                         # q missing


def test_ops_validate_on_host():
    torch = pytest.importorskip("torch")
    from pto_fuser_amd import gdn_chunk_forward, kkt_inverse, tri_inv
    q = torch.zeros(1, 1, 64, 128)
    with pytest.raises(ValueError, match="HIP device"):
        gdn_chunk_forward(q, q, q, torch.zeros(1, 1, 64))
    with pytest.raises(ValueError, match="multiple of the chunk"):
        gdn_chunk_forward(torch.zeros(1, 1, 65, 128), q, q, torch.zeros(1, 1, 65))
    with pytest.raises(ValueError, match="unsupported shape"):
        gdn_chunk_forward(torch.zeros(1, 1, 64, 64), q, q, torch.zeros(1, 1, 64))
    with pytest.raises(ValueError):
        tri_inv(torch.zeros(2, 64, 32))
    with pytest.raises(ValueError):
        kkt_inverse(torch.zeros(64, 128), None, torch.zeros(64), chunk_size=32)
    from pto_fuser_amd import kda_chunk_forward
    qb = torch.zeros(1, 1, 128, 128, dtype=torch.bfloat16)
    gk = torch.zeros(1, 1, 128, 128)
    with pytest.raises(ValueError, match="HIP device"):
        kda_chunk_forward(qb, qb, qb, torch.zeros(1, 1, 128), gk)
    with pytest.raises(ValueError, match="bfloat16 or float32"):
        kda_chunk_forward(qb.half(), qb.half(), qb.half(), torch.zeros(1, 1, 128), gk)
    with pytest.raises(ValueError, match="multiple of the chunk size"):
        kda_chunk_forward(qb[:, :, :96], qb[:, :, :96], qb[:, :, :96], torch.zeros(1, 1, 96), gk[:, :, :96])


@pytest.mark.parametrize("device", [None, 0, "cuda", "cuda:0", torch.device("cuda"), torch.device("cuda:0")])
def test_stream_handle_of_every_device_form(monkeypatch, device):
    """A device given as a string or an index names the same stream as the torch.device does; a CPU device
    with an index does not pass for the GPU of that index."""
    class Stream:
        cuda_stream = 7

    def current_stream(dev=None):
        if dev is not None and not isinstance(dev, int) and torch.device(dev).type != "cuda":
            raise ValueError(f"Expected a cuda device, but got: {dev}")
        return Stream

    monkeypatch.setattr(torch.cuda, "current_stream", current_stream)
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda index: 7 + int(index), raising=False)
    assert _hip.current_stream_handle(device) == 7
    with pytest.raises(ValueError):
        _hip.current_stream_handle(torch.device("cpu", 0))


@pytest.mark.parametrize("name", ["gdn", "kda"])
def test_workspaces_of_every_device_form(monkeypatch, name):
    """A workspace can be asked for by device, string, index or None (the current device); the forms that
    name one device share it."""
    from pto_fuser_amd import ops
    made = []

    class Fake:
        def __init__(self, *args):
            made.append(args[-1])

        def close(self):
            pass

    monkeypatch.setattr(ops, name.capitalize() + "Workspace", Fake)
    monkeypatch.setattr(ops, "_WORKSPACES", {})
    monkeypatch.setattr(ops._hip, "current_stream_handle", lambda device=None: 7)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    get = getattr(ops, name + "_workspace")
    one = [get(1, 1, 64, 64, 128, 128, torch.float32, dev) for dev in ("cuda:0", 0, torch.device("cuda", 0))]
    assert one[0] is one[1] is one[2]
    current = get(1, 1, 64, 64, 128, 128, torch.float32, None)
    assert isinstance(current, Fake) and made == [torch.device("cuda:0"), None]
