"""The C-ABI library loads and exports every symbol include/iron_hip.h declares (no GPU needed)."""

import ctypes
import re
from pathlib import Path

import pytest

from iron_amd import _lib

ROOT = Path(__file__).resolve().parent.parent


def declared_symbols():
    text = (ROOT / "include" / "iron_hip.h").read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(iron_[a-z0-9_]+)\s*\(", text)))


def test_header_and_binding_agree():
    assert declared_symbols() == sorted(_lib.SIGNATURES)


def test_library_exports_every_declared_symbol():
    handle = ctypes.CDLL(str(_lib.LIB_PATH))
    for name in declared_symbols():
        assert hasattr(handle, name), name
    lib = _lib.lib()
    assert lib.iron_version() >= 100
    assert lib.iron_mha_decode_workspace_bytes(32, 64) == 32 * 128 * 66 * 4


def test_argument_refusals_need_no_gpu():
    """A refused call returns 1 before any launch and leaves its reason readable."""
    lib = _lib.lib()
    assert lib.iron_gemv_bf16(None, None, None, 8, 8, 1, 1, None, None) == 1
    assert b"null operand" in lib.iron_last_error()
    one = ctypes.c_void_p(16)
    assert lib.iron_gemv_bf16(one, one, one, 8, 12, 1, 1, None, None) == 1
    assert b"multiple of 8" in lib.iron_last_error()
    assert lib.iron_mha_prefill_bf16(one, one, one, one, 6, 4, 64, 8, 8, 8, 0.125, 1, -1, 0, 0, None, None, None) == 1
    assert b"multiple of kv_heads" in lib.iron_last_error()
    for name, operands in (("gemm_gated_pair", 5), ("gemm_gated_product", 4)):   # (two entry points of one function)
        call = getattr(lib, f"iron_{name}_bf16")
        for sizes, why in (((64, 64, 64, 0), b"activation"), ((64, 64, 40, 1), b"multiple of 64"), ((64, 1 << 23, 64, 1), b"at most 2^22")):
            assert call(*(ctypes.c_void_p(16 * i + 16) for i in range(operands)), *sizes, None, None) == 1
            assert lib.iron_last_error().startswith(name.encode() + b":") and why in lib.iron_last_error()


def test_every_entry_point_refuses_null_operands():
    """Each entry point that takes pointers returns 1 with a reason, before any launch, when they
    are all null and every size is zero: nothing is dereferenced or launched on bad arguments."""
    lib = _lib.lib()
    for name, (_, args) in sorted(_lib.SIGNATURES.items()):
        if not any(a is _lib._P for a in args):
            continue
        call = [None if a is _lib._P else (0.0 if a is ctypes.c_float else 0) for a in args]
        assert getattr(lib, name)(*call) == 1, name
        assert lib.iron_last_error(), name


def test_a_latent_step_s_splits():
    """As many as fill the chip: of blocks of sixteen heads in bf16, of twice as many of one head in float32 and in bf16 of sizes for any."""
    room = _lib.lib().iron_mha_latent_workspace_bytes
    for slots, heads, rank, rot, window, is_float, splits in ((16, 2, 1024, 0, 2048, 1, 32), (16, 2, 1024, 0, 2048, 0, 16), (16, 2, 1023, 0, 2048, 0, 32),
                                                              (4, 16, 512, 64, 4096, 1, 64), (64, 33, 512, 64, 4096, 0, 8), (1, 4, 512, 64, 100, 1, 2)):
        absorbed = -(-slots * heads * (rank + rot) * 4 // 16) * 16
        sums = -(-slots * splits * heads * rank * 4 // 16) * 16
        assert room(slots, slots, heads, 128, rot, 128, rank, window, window, 0, 1, is_float) == absorbed + sums + slots * splits * heads * 8


def test_few_rows_over_a_long_k_share_no_tiles():
    """Up to sixteen rows against up to 2048 of a long K go by strips, whatever the product of rows and K; past that, and past
    K = 16384, their tiles' K is dealt over blocks where that takes less than the few rows would.  As (N,M) output the same with the operands' places changed."""
    room = _lib.lib().iron_gemm_workspace_bytes
    for M, N, K, shared in ((16, 2048, 9216, False), (9, 1536, 16384, False), (16, 304, 14336, False), (16, 128, 16384, False),
                            (16, 120, 16384, True), (16, 2056, 9216, True), (17, 2048, 9216, True), (12, 2048, 16392, True),
                            (16, 4096, 10192, False), (40, 2048, 8192, True), (45, 512, 8184, True)):
        assert (room(M, N, K, 1, 0) > 0) == shared, (M, N, K)
        assert (room(N, M, K, 1, 1) > 0) == shared, (N, M, K)


def test_a_product_of_one_round_of_small_tiles_takes_them_or_shares_its_k():
    """Up to 64 rows or columns against as many of the other as make 128 tiles of 128 x 128: where sharing a long K is given up because
    small tiles are the cheaper, the launch takes small tiles, in every layout and up to the last column."""
    lib = _lib.lib()
    for K in (1024, 4096, 6200, 8192, 12288):
        for few in (33, 64):
            for many in (8192, 16256, 16264, 16320, 16384):
                for M, N, b, c in ((few, many, 0, 0), (many, few // 8 * 8, 0, 0), (few, many, 0, 1), (many, few // 8 * 8, 0, 1), (many, 32, 1, 0), (32, many, 1, 1)):
                    tile, room = lib.iron_gemm_tile(0, M, N, K, b, c, 0), lib.iron_gemm_workspace_bytes(M, N, K, b, c)
                    assert tile in (32 << 16 | 64, 64 << 16 | 64, 64 << 16 | 32, 32 << 16 | 32, 0), (M, N, K, b, c, tile >> 16, tile & 65535, room)
    assert lib.iron_gemm_workspace_bytes(64, 16384, 8192, 0, 0) == 0 and lib.iron_gemm_tile(0, 64, 16384, 8192, 0, 0, 0) == 64 << 16 | 64


def test_few_rows_of_a_matrix_from_memory_share_its_k():
    """With B (K,N) of more than 16 MB a tile of 64 columns draws a line of each row out of memory: too few of them to fill the chip share K instead, in
    either order of C; a matrix that the caches hold, or one of more columns over a shorter K, stays on small tiles."""
    room = _lib.lib().iron_gemm_workspace_bytes
    for M, N, K, c, shared in ((59, 6144, 4712, 0, True), (1, 5120, 4336, 1, True), (9, 6144, 3824, 0, True), (1, 5120, 4088, 0, True), (10, 4096, 3776, 0, True),
                               (10, 12288, 2736, 0, False), (16, 6144, 1024, 0, False), (130, 72, 2504, 0, True), (29, 6144, 2040, 0, False), (8, 1024, 4096, 0, True)):
        assert (room(M, N, K, 0, c) > 0) == shared, (M, N, K)


def test_short_products_under_a_bound_take_large_tiles_for_many_rows():
    """Up to K = 1536 a round of tiles is mostly its start and its end: rows that make several rounds of 64 x 64 tiles take larger ones, fewer
    of a product whose second operand its epilogue reads than of a plain one."""
    tile = _lib.lib().iron_gemm_tile
    for kind, M, N, K, want in ((1, 2048, 2560, 64, (192, 128)), (1, 2048, 3064, 64, (256, 128)), (1, 2048, 6144, 512, (256, 256)), (1, 2048, 1280, 128, (128, 128)),
                                (2, 2048, 2560, 64, (192, 128)), (2, 2048, 1256, 128, (128, 128)), (2, 2048, 6144, 512, (128, 128)), (2, 256, 8376, 64, (128, 128)),
                                (1, 1024, 4552, 192, (160, 128)), (2, 64, 26574, 1152, (128, 128)), (2, 64, 32000, 1216, (128, 128)), (1, 4, 20111, 1056, (128, 128))):
        got = tile(kind, M, N, K, 1, 0, M)
        assert (got >> 16, got & 65535) == want, (kind, M, N, K, got >> 16, got & 65535)
    # (two 64 x 64 tiles a CU: few tiles of a short K whatever the bound, of a longer one without a bound)
    for kind, M, N, K, rows, want in ((1, 2048, 672, 192, 670, (64, 64)), (2, 2048, 528, 256, 0, (64, 64)), (2, 2048, 528, 512, 0, (64, 64)), (2, 2048, 624, 1024, 0, (64, 64)),
                                      (2, 2048, 528, 512, 2048, (128, 64)), (2, 1024, 1904, 1024, 0, (128, 64)), (2, 2048, 568, 960, 119, (32, 32)),
                                      (1, 64, 28672, 192, 3, (64, 64)), (2, 64, 19760, 128, 64, (64, 64)), (1, 40, 36000, 960, 33, (64, 64))):
        got = tile(kind, M, N, K, 1, 0, rows)
        assert (got >> 16, got & 65535) == want, (kind, M, N, K, rows, got >> 16, got & 65535)
    for kind in (1, 2):   # (and few rows small ones)
        for K in (64, 448, 512, 1024):
            assert tile(kind, 2048, 1024, K, 1, 0, 40) in (64 << 16 | 64, 64 << 16 | 32, 32 << 16 | 32)


def test_large_products_without_a_bound_reach_every_size_of_tile():
    """The sizes at which the GPU's tests take each large tile for their own, by what the launch chooses."""
    tile = _lib.lib().iron_gemm_tile
    for want, sizes in {(256, 256): [(3329, 128, 3593, 1, 0), (3329, 192, 3592, 0, 0)], (192, 256): [(192, 136, 48000, 1, 0), (3840, 264, 2819, 1, 0), (1290, 200, 8200, 0, 0)],
                        (160, 256): [(160, 200, 40963, 1, 0), (1025, 64, 7169, 1, 0), (1025, 72, 7176, 0, 0)],
                        (128, 256): [(641, 264, 8067, 1, 0), (777, 64, 6915, 1, 0), (641, 136, 5384, 0, 0)],
                        (128, 192): [(128, 328, 33000, 1, 0), (641, 64, 5377, 1, 0), (3585, 200, 1025, 1, 1)]}.items():
        for M, K, N, b, c in sizes:
            got = tile(0, M, N, K, b, c, 0)
            assert (got >> 16, got & 65535) == want, (M, K, N, b, c)
    for M, N, K in ((8192, 1400, 1608), (32000, 1040, 3904), (749, 26520, 4912), (17071, 1384, 1384), (1274, 19568, 1976)):   # B (K,N), where 128 x 128 tiles take more than their price
        assert tile(0, M, N, K, 0, 0, 0) != 128 << 16 | 128, (M, N, K)


def test_few_rows_go_by_long_stages_where_a_launch_has_the_blocks():
    """Up to 32 rows over whole 256 of K, eight columns a block (32 of each of a pair): as many blocks as the buffer's most rows have tiles, so a buffer of few rows
    has too few for many columns; not a K of other lengths, nor more rows, nor more columns than CUs have room for."""
    tile = _lib.lib().iron_gemm_tile
    for kind, M, N, K, rows, long in ((1, 600, 2048, 2048, 32, 8), (1, 600, 2048, 2048, 33, 0), (1, 64, 2048, 2048, 32, 0), (1, 64, 1024, 2048, 32, 0), (1, 128, 2048, 2048, 32, 8),
                                      (2, 600, 2048, 8192, 1, 8), (2, 600, 2056, 8192, 1, 0), (1, 600, 2048, 2112, 32, 0), (1, 600, 2044, 2048, 32, 0),
                                      (3, 64, 8192, 2048, 32, 32), (3, 600, 8192, 2048, 32, 32), (3, 600, 8192, 2048, 33, 0), (3, 600, 8200, 2048, 32, 0), (3, 600, 8192, 2112, 9, 0),
                                      (0, 17, 4096, 2048, 0, 16), (0, 16, 4096, 2048, 0, 0), (0, 33, 4096, 2048, 0, 0)):
        got = tile(kind, M, N, K, 1, 0, rows)
        assert (got & 32767 if got >> 15 & 1 else 0) == long, (kind, M, N, K, rows, hex(got))


def test_what_a_bound_chooses_is_decided_once_for_the_same_sizes():
    """A launch under a row bound prices every form for every run of rows: the same sizes again cost no more than a launch without a bound,
    and more sizes than are held, or another thread, change no answer."""
    import threading
    import time

    tile = _lib.lib().iron_gemm_tile

    def best(*args):
        times = []
        for _ in range(9):
            start = time.perf_counter()
            for _ in range(300):
                tile(*args)
            times.append(time.perf_counter() - start)
        return min(times)

    assert best(1, 4096, 2048, 2048, 1, 0, 1000) < 2 * best(0, 4096, 2048, 2048, 1, 0, 0)
    asked = [(kind, M, N, K, 1, 0, rows) for kind in (1, 2, 3) for M in (300, 2048, 4096, 5000) for N in (2048, 2056, 8192) for K in (448, 2048)
             for rows in (1, 130, 300, 2048)]
    first, again = [tile(*a) for a in asked], []
    other = threading.Thread(target=lambda: again.extend(tile(*a) for a in reversed(asked)))
    other.start()
    other.join()
    assert first == again[::-1] == [tile(*a) for a in asked] and len(set(first)) > 6


def test_bench_refuses_more_than_one_gpu():
    """``bench.py --gpus N`` with N above 1 exits with a message: this build is the one-GPU path."""
    import subprocess
    import sys
    from pathlib import Path

    bench = Path(__file__).resolve().parent.parent / "bench.py"
    done = subprocess.run([sys.executable, str(bench), "--gpus", "2"], capture_output=True, text=True, timeout=120)
    assert done.returncode != 0 and "one-GPU" in done.stderr and done.stdout.strip() == ""


def test_native_calls_leave_what_is_not_plain_to_the_caller():
    """The one-call shortcut answers None, and raises nothing, for tensors off the GPU, other types of number and of argument, and
    counts past 32 bits; the operators' own words are then what a caller reads."""
    import torch

    from iron_amd import kernels as K
    from iron_amd._lib import native

    a = torch.zeros(8, 8, dtype=torch.bfloat16)
    for args in ((a, a, a, 8, 8, 8, True, False), (None, a, a, 8, 8, 8, 0, 0), (a, a, a, 8.0, 8, 8, 0, 0), (a, a, a, 1 << 40, 8, 8, 0, 0),
                 (a, a, a, 8, 8, 8, "x", 0), (a, a, a, 8, 8)):
        assert native().gemm(*args) is None
    assert native().gemv(a, a, a, 8, 8) is None and native().gemv(a) is None
    assert native().mha_prefill(a, a, a, a, 1.0, 1, 1, 64, -8, 8, 8, 1, -1, 0, 0) is None and native().mha_prefill(a) is None
    with pytest.raises(TypeError, match="A: expected a tensor on the GPU"):
        K.gemm(a, a, a, M=8, N=8, K=8)
    with pytest.raises(TypeError, match="expected a torch tensor"):
        K.gemv([1.0], a, a, M=8, K=8)


def test_operators_go_the_long_way_where_the_native_calls_do_not_load(monkeypatch):
    """A tree without ``_calls``, or with one built for another torch: one warning, and the operators' own words for what they refuse."""
    import sys
    import warnings

    import torch

    import iron_amd
    from iron_amd import kernels as K

    monkeypatch.setitem(sys.modules, "iron_amd._calls", None)   # an import of it raises ImportError
    monkeypatch.delattr(iron_amd, "_calls", raising=False)
    _lib.native.cache_clear()
    try:
        a = torch.zeros(8, 8, dtype=torch.bfloat16)
        with pytest.warns(RuntimeWarning, match="iron_amd._calls does not load"), pytest.raises(TypeError, match="A: expected a tensor on the GPU"):
            K.gemm(a, a, a, M=8, N=8, K=8)
        with warnings.catch_warnings():
            warnings.simplefilter("error")
            for call in (lambda: K.gemv(a, a, a, M=8, K=8), lambda: K.mha_prefill(a, a, a, a, heads=1, kv_heads=1, d=64, seq=1, kv_len=1)):
                with pytest.raises(TypeError, match="expected a tensor on the GPU"):
                    call()
    finally:
        _lib.native.cache_clear()


def test_the_library_is_linked_where_the_native_calls_are_not_built(monkeypatch, tmp_path):
    """A build whose native calls fail leaves the library, leaves no native calls of another build beside it, and says what failed."""
    from iron_amd import build

    (tmp_path / "csrc").mkdir()
    (tmp_path / "csrc" / "calls.cpp").write_text("#error no headers")
    (tmp_path / "csrc" / "one.hip").write_text("")
    (tmp_path / "_calls.so").write_text("another build's")
    ran = []

    def run(cmd):
        ran.append(cmd)
        if any(str(c).endswith("calls.cpp") for c in cmd):
            raise RuntimeError("no headers")
        Path(cmd[cmd.index("-o") + 1]).write_text("built")

    for name, value in (("HERE", tmp_path), ("CSRC", tmp_path / "csrc"), ("LIB", tmp_path / "lib.so"), ("CALLS", tmp_path / "_calls.so"), ("_run", run),
                        ("_hipcc", lambda: "hipcc")):
        monkeypatch.setattr(build, name, value)
    with pytest.raises(RuntimeError, match="no headers"):
        build.build()
    assert (tmp_path / "lib.so").read_text() == "built" and not (tmp_path / "_calls.so").exists()
    assert all(cmd[0] == "hipcc" for cmd in ran)
