"""CPU-only checks of the C ABI: the library loads, exports what include/ring_attention_hip.h
declares, rejects bad arguments before touching a GPU, and classifies skippable ring steps
exactly like a brute-force evaluation of the bias."""
import ctypes as C
import os
import re

import numpy as np
import pytest

from oracle import ring_oracle as R
from ring_attention import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "ring_attention_hip.h")


def _declared():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(ra_[a-z_0-9]+)\s*\(", text)))


def test_library_exports_every_declared_symbol(lib):
    names = _declared()
    assert len(names) >= 12
    for n in names:
        assert hasattr(lib, n), f"{n} declared in the header but not exported"
    assert sorted(_lib.EXPORTS) == names, "python binding table and header disagree"
    assert lib.ra_version() >= 1000


def test_struct_layout_matches_header():
    # sizes implied by the header with natural alignment on x86-64
    assert C.sizeof(_lib.RaTensor) == 32
    assert C.sizeof(_lib.RaBias) == 8 + 16 + 16 + 16 + 16 + 16 + 8 + 8 + 24 + 8
    assert C.sizeof(_lib.RaFwdStepParams) == 24 + 3 * 32 + 24 + C.sizeof(_lib.RaBias)
    assert C.sizeof(_lib.RaBwdStepParams) == 24 + 4 * 32 + 40 + C.sizeof(_lib.RaBias)


def _good_fwd():
    p = _lib.RaFwdStepParams()
    p.B, p.H, p.Lq, p.Lk, p.D = 1, 2, 64, 64, 128
    p.sm_scale = 0.1
    for t in (p.q, p.k, p.v):
        t.ptr, t.stride_b, t.stride_h, t.stride_l = 0x1000, 64 * 256, 128, 256
    p.o = p.m = p.l = 0x2000
    return p


def _good_bwd():
    p = _lib.RaBwdStepParams()
    p.B, p.H, p.Lq, p.Lk, p.D = 1, 2, 64, 64, 64
    p.sm_scale = 0.1
    for t in (p.q, p.k, p.v, p.dout):
        t.ptr, t.stride_b, t.stride_h, t.stride_l = 0x1000, 64 * 128, 64, 128
    p.lse = p.delta = p.dq = p.dk = p.dv = 0x2000
    return p


def test_check_accepts_good_params(lib):
    assert lib.ra_fwd_step_check(C.byref(_good_fwd())) == 0
    assert lib.ra_bwd_step_check(C.byref(_good_bwd())) == 0


@pytest.mark.parametrize("mutate,code", [
    (lambda p: setattr(p, "D", 96), -3),
    (lambda p: setattr(p, "D", 256), -3),
    (lambda p: setattr(p, "Lq", 0), -2),
    (lambda p: setattr(p, "B", -1), -2),
    (lambda p: setattr(p.q, "ptr", None), -1),
    (lambda p: setattr(p.k, "ptr", 0x1008), -4),
    (lambda p: setattr(p.v, "stride_l", 129), -4),
    (lambda p: setattr(p, "o", None), -1),
    (lambda p: setattr(p, "sm_scale", float("nan")), -2),
    (lambda p: setattr(p.bias, "flags", 64), -5),
    (lambda p: setattr(p.bias, "flags", _lib.RA_BIAS_WINDOW), -5),            # window == 0
    (lambda p: setattr(p.bias, "flags", _lib.RA_BIAS_CAUSAL | _lib.RA_BIAS_PREFIX), -5),
    (lambda p: setattr(p.bias, "flags", _lib.RA_BIAS_SEGMENT), -1),           # no id arrays
    (lambda p: setattr(p.bias, "flags", _lib.RA_BIAS_ALIBI), -1),             # no slopes
    (lambda p: setattr(p.bias, "flags", _lib.RA_BIAS_DENSE), -1),             # no dense block
    (lambda p: (setattr(p.bias, "flags", _lib.RA_BIAS_DENSE), setattr(p.bias, "dense_bias", 0x3000),
                setattr(p.bias, "dense_stride_q", 63)), -5),                  # rows overlap
    (lambda p: (setattr(p.bias, "flags", _lib.RA_BIAS_DENSE), setattr(p.bias, "dense_bias", 0x3002),
                setattr(p.bias, "dense_stride_q", 64)), -4),
    (lambda p: (setattr(p.bias, "flags", _lib.RA_BIAS_CAUSAL), setattr(p.bias, "q_offset", -5)), -5),
    # positions (offset + index) stay below RA_MAX_POSITION: the last token of the shard counts
    (lambda p: (setattr(p.bias, "flags", _lib.RA_BIAS_CAUSAL),
                setattr(p.bias, "q_offset", _lib.RA_MAX_POSITION - p.Lq + 1)), -5),
    (lambda p: (setattr(p.bias, "flags", _lib.RA_BIAS_CAUSAL),
                setattr(p.bias, "kv_offset", _lib.RA_MAX_POSITION - p.Lk + 1)), -5),
])
def test_fwd_step_rejects_bad_params_without_a_gpu(lib, mutate, code):
    p = _good_fwd()
    mutate(p)
    assert lib.ra_fwd_step_check(C.byref(p)) == code
    assert lib.ra_fwd_step(C.byref(p), None) == code  # validation comes before any HIP call
    assert lib.ra_last_error() != b""


def test_position_and_window_limits(lib):
    # the largest positions and any window width pass the checks (a window wider than every
    # position difference masks nothing and is clamped inside the library)
    p = _good_fwd()
    p.bias.flags = _lib.RA_BIAS_CAUSAL | _lib.RA_BIAS_WINDOW
    p.bias.window = 2 ** 31 - 1
    p.bias.q_offset = _lib.RA_MAX_POSITION - p.Lq
    p.bias.kv_offset = _lib.RA_MAX_POSITION - p.Lk
    assert lib.ra_fwd_step_check(C.byref(p)) == 0
    # a step against keys 2^30 positions behind a window of 2^31 - 1 still has work; one beyond a
    # small window has none
    p.bias.kv_offset = 0
    assert lib.ra_step_is_skippable(C.byref(p.bias), p.Lq, p.Lk) == 0
    p.bias.window = 1000
    assert lib.ra_step_is_skippable(C.byref(p.bias), p.Lq, p.Lk) == 1


def test_row_stride_limits(lib):
    # rows may not overlap (stride_l >= D) and the row stride stays within 2^27 elements: the kernels
    # reach the rows one wavefront moves through a 32-bit byte offset from the wavefront's first row
    for bad in (0, -128, 64, _lib.RA_MAX_ROW_STRIDE + 8):
        p = _good_fwd()
        p.k.stride_l = bad
        assert p.D == 128 and lib.ra_fwd_step_check(C.byref(p)) == -2, bad
        assert b"row stride" in lib.ra_last_error()
        p = _good_bwd()
        p.dout.stride_l = min(bad, 56)  # D = 64 there
        assert lib.ra_bwd_step_check(C.byref(p)) == -2, bad
    for good in (128, 136, _lib.RA_MAX_ROW_STRIDE):
        p = _good_fwd()
        p.v.stride_l = good
        assert lib.ra_fwd_step_check(C.byref(p)) == 0, good


def test_dense_map_arguments_are_checked_without_a_gpu(lib):
    """ra_dense_map_bytes is plain arithmetic; ra_dense_map and a step that carries a summary
    refuse bad arguments before anything is launched."""
    assert lib.ra_dense_map_bytes(0, 0, 2, 3, 64, 64) == 4
    assert lib.ra_dense_map_bytes(1 << 20, 0, 2, 3, 100, 250) == 2 * 4 * 8
    assert lib.ra_dense_map_bytes(1 << 20, 1 << 16, 2, 3, 33, 1031) == 2 * 3 * 2 * 33
    assert lib.ra_dense_map_bytes(0, 0, 0, 3, 64, 64) == 0
    good = dict(dense_bias=0x1000, stride_b=0, stride_h=0, stride_q=64, B=1, H=1, Lq=64, Lk=64, map=0x2000)

    def call(**kw):
        a = {**good, **kw}
        return lib.ra_dense_map(a["dense_bias"], a["stride_b"], a["stride_h"], a["stride_q"], a["B"], a["H"],
                                a["Lq"], a["Lk"], a["map"], None)

    assert call(dense_bias=None) == -1 and call(map=None) == -1          # RA_ERR_NULL
    assert call(Lq=0) == -2 and call(B=-1) == -2                          # RA_ERR_SHAPE
    assert call(Lk=_lib.RA_MAX_SEGMENT_SHARD + 1, stride_q=1 << 20) == -2
    assert call(dense_bias=0x1002) == -4                                  # RA_ERR_ALIGN
    assert call(stride_q=63) == -5 and call(stride_b=-8) == -5            # RA_ERR_BIAS
    # a step whose dense block comes with a summary: shards of at most RA_MAX_SEGMENT_SHARD tokens
    p = _good_fwd()
    p.bias.flags = _lib.RA_BIAS_DENSE
    p.bias.dense_bias, p.bias.dense_stride_q, p.bias.dense_map = 0x3000, 64, 0x4000
    assert lib.ra_fwd_step_check(C.byref(p)) == 0
    p.Lk = _lib.RA_MAX_SEGMENT_SHARD + 64
    p.bias.dense_stride_q = p.Lk
    assert lib.ra_fwd_step_check(C.byref(p)) == -2 and b"summary" in lib.ra_last_error()
    p.bias.dense_map = None
    assert lib.ra_fwd_step_check(C.byref(p)) == 0


def test_bwd_step_rejects_bad_params_without_a_gpu(lib):
    p = _good_bwd()
    p.dk = None
    assert lib.ra_bwd_step(C.byref(p), None) == -1
    p = _good_bwd()
    p.dout.stride_h = 3
    assert lib.ra_bwd_step(C.byref(p), None) == -4
    p = _good_bwd()
    assert lib.ra_bwd_step_parts(C.byref(p), 7, None) == -2
    assert lib.ra_fwd_step(None, None) == -1
    assert lib.ra_fwd_init(None, None, None, 1, 1, 1, 64, None) == -1
    assert lib.ra_fwd_finalize(0x10, 0x10, 0x10, 0x10, 5, 8, 8, 8, 0x10, 1, 1, 1, 64, None) == -7


def test_finalize_entry_points_check_alignment_without_a_gpu(lib):
    # ra_fwd_finalize stores four elements at a time: out must be aligned to 8 (bf16) / 16 (fp32) bytes
    ok = (0x1000, 0x1000, 0x1000)
    assert lib.ra_fwd_finalize(*ok, 0x2004, _lib.RA_DTYPE_BF16, 128, 128, 128, 0x3000, 1, 1, 4, 64, None) == -4
    assert b"aligned" in lib.ra_last_error()
    assert lib.ra_fwd_finalize(*ok, 0x2008, _lib.RA_DTYPE_F32, 128, 128, 128, 0x3000, 1, 1, 4, 64, None) == -4
    assert lib.ra_fwd_finalize(0x1004, 0x1000, 0x1000, 0x2000, _lib.RA_DTYPE_F32, 128, 128, 128, 0x3000,
                               1, 1, 4, 64, None) == -4
    assert lib.ra_fwd_finalize(*ok, 0x2000, _lib.RA_DTYPE_F32, 130, 128, 128, 0x3000, 1, 1, 4, 64, None) == -4
    # ra_bwd_finalize loads 16 bytes of fp32 and stores 8 bytes of bf16 at a time
    assert lib.ra_bwd_finalize(0x1000, 0x2004, 128, 128, 128, 1, 1, 4, 64, None) == -4
    assert b"8-byte" in lib.ra_last_error()
    assert lib.ra_bwd_finalize(0x1008, 0x2000, 128, 128, 128, 1, 1, 4, 64, None) == -4
    assert lib.ra_bwd_finalize(0x1000, 0x2000, 128, 126, 128, 1, 1, 4, 64, None) == -4


def test_grids_beyond_the_launch_limit_are_rejected(lib):
    # B*H*ceil(L/128) workgroups must fit a 31-bit grid dimension: a larger launch would be cut short
    p = _good_fwd()
    p.B, p.H, p.Lq = 1 << 10, 1 << 10, 1 << 22      # 2^20 heads x 2^15 tiles = 2^35 workgroups
    assert lib.ra_fwd_step_check(C.byref(p)) == -2 and b"grid" in lib.ra_last_error()
    p.Lq, p.Lk = 64, 1 << 22                          # the key side counts as well (dK/dV grid)
    assert lib.ra_fwd_step_check(C.byref(p)) == -2
    b = _good_bwd()
    b.B, b.H, b.Lk = 1 << 10, 1 << 10, 1 << 22
    assert lib.ra_bwd_step_check(C.byref(b)) == -2
    p = _good_fwd()
    p.B, p.H, p.Lq = 1 << 10, 1 << 10, 1 << 17      # 2^30 workgroups: still fine
    assert lib.ra_fwd_step_check(C.byref(p)) == 0


@pytest.mark.parametrize("flags,window", [(1, 0), (3, 7), (2, 7), (3, 64), (2, 1), (0, 0), (8, 0)])
def test_step_is_skippable_matches_brute_force(lib, flags, window):
    Lq, Lk = 16, 24
    for q_off in (0, 16, 40, 100):
        for kv_off in (0, 24, 48, 96):
            b = _lib.RaBias()
            b.flags, b.window, b.q_offset, b.kv_offset = flags, window, q_off, kv_off
            got = lib.ra_step_is_skippable(C.byref(b), Lq, Lk)
            qp = (q_off + np.arange(Lq))[None]
            kp = (kv_off + np.arange(Lk))[None]
            fn = R.make_bias_fn(causal=bool(flags & 1), window=window if flags & 2 else None,
                                use_prefix=bool(flags & 8))
            pm_q = np.ones((1, Lq), dtype=np.int32); pm_k = np.ones((1, Lk), dtype=np.int32)
            bias = fn(q_positions=qp, kv_positions=kp, q_prefix_mask=pm_q, kv_prefix_mask=pm_k)
            want = int(np.all(np.isneginf(bias)))
            if flags & 8:
                want = 0  # prefix masks are data dependent: never skipped on the host
            assert got == want, (flags, window, q_off, kv_off)


def _steps(make, n):
    arr = (type(make()) * n)()
    for i in range(n):
        arr[i] = make()
    return arr


def test_multi_step_entry_points_validate_before_any_gpu_call(lib):
    # nothing to do / bad counts
    assert lib.ra_fwd_steps(None, 0, None) == 0
    assert lib.ra_fwd_steps(None, 2, None) == -1
    assert lib.ra_bwd_dq_steps(None, -1, None) == -2
    assert lib.ra_bwd_dkdv_steps(None, 3, None) == -1
    # every block goes through the single-step checks
    f = _steps(_good_fwd, 3)
    f[2].D = 96
    assert lib.ra_fwd_steps(f, 3, None) == -3
    # the blocks of one launch may differ in the travelling shard only
    f = _steps(_good_fwd, 2)
    f[1].o = 0x3000
    assert lib.ra_fwd_steps(f, 2, None) == -2 and b"steps[1]" in lib.ra_last_error()
    f = _steps(_good_fwd, 2)
    f[1].k.stride_l = 512
    assert lib.ra_fwd_steps(f, 2, None) == -2
    f = _steps(_good_fwd, 2)
    f[1].bias.q_offset = 64
    assert lib.ra_fwd_steps(f, 2, None) == -2
    b = _steps(_good_bwd, 2)
    b[1].lse = 0x4000          # the query side is fixed in a dq launch ...
    assert lib.ra_bwd_dq_steps(b, 2, None) == -2
    b = _steps(_good_bwd, 2)
    b[1].dk = 0x4000           # ... and the key/value side in a dk/dv launch
    assert lib.ra_bwd_dkdv_steps(b, 2, None) == -2
    b = _steps(_good_bwd, 2)
    b[1].bias.kv_offset = 64
    assert lib.ra_bwd_dkdv_steps(b, 2, None) == -2
    # steps that are masked entirely are dropped on the host: nothing is launched for these
    for arr, fn in ((_steps(_good_fwd, 2), lib.ra_fwd_steps), (_steps(_good_bwd, 2), lib.ra_bwd_dq_steps),
                    (_steps(_good_bwd, 2), lib.ra_bwd_dkdv_steps)):
        for p in arr:
            p.bias.flags = _lib.RA_BIAS_CAUSAL
            p.bias.kv_offset = 1 << 20
        assert fn(arr, 2, None) == 0


def _pair_fwd(lib, mutate=None, **kw):
    p = _good_fwd()
    p.o = p.m = p.l = None  # not used
    if mutate:
        mutate(p)
    a = {**dict(out=0x1000, dtype=_lib.RA_DTYPE_BF16, sb=64 * 256, sh=128, sl=256, lse=0x2000, ws=0x3000, size=1 << 30), **kw}
    return lib.ra_fwd_pair(C.byref(p), a["out"], a["dtype"], a["sb"], a["sh"], a["sl"], a["lse"], a["ws"], a["size"], None)


def test_fwd_pair_rejects_bad_arguments_without_a_gpu(lib):
    def long(p):  # 1 x 2 heads of 64 rows against 4096 keys: shared by several workgroups
        p.Lk = 4096

    assert lib.ra_fwd_pair(None, 0x1000, 0, 8, 8, 8, 0x2000, None, 0, None) == -1
    for kw, code in ((dict(out=None), -1), (dict(lse=None), -1), (dict(dtype=5), -7), (dict(dtype=_lib.RA_DTYPE_F16), -7),
                     (dict(out=0x1004), -4), (dict(out=0x1008, dtype=_lib.RA_DTYPE_F32), -4), (dict(sl=254), -4),
                     (dict(mutate=lambda p: setattr(p, "D", 96)), -3), (dict(mutate=lambda p: setattr(p.k, "ptr", None)), -1),
                     (dict(mutate=lambda p: setattr(p.bias, "flags", 64)), -5),
                     (dict(mutate=long, ws=None), -4), (dict(mutate=long, ws=0x3008), -4), (dict(mutate=long, size=1000), -2)):
        assert _pair_fwd(lib, **kw) == code, kw
        assert lib.ra_last_error() != b""
    p = _good_fwd()
    assert lib.ra_fwd_pair_workspace(C.byref(p)) == 0
    long(p)
    size = lib.ra_fwd_pair_workspace(C.byref(p))
    assert size > 0 and size % 4 == 0
    assert _pair_fwd(lib, mutate=long, size=size - 1) == -2
    p.D = 96
    assert lib.ra_fwd_pair_workspace(C.byref(p)) == 0 and lib.ra_fwd_pair_workspace(None) == 0


def test_bwd_pair_rejects_bad_arguments_without_a_gpu(lib):
    good = dict(out=0x1000, dtype=_lib.RA_DTYPE_BF16, os=(64 * 128, 64, 128), dq=0x4000, qs=(64 * 128, 64, 128), dk=0x5000, dv=0x6000,
                ks=(64 * 128, 64, 128), ws=0x7000, size=1 << 30)

    def call(mutate=None, **kw):
        p = _good_bwd()
        p.delta = p.dq = p.dk = p.dv = None  # not used
        if mutate:
            mutate(p)
        a = {**good, **kw}
        return lib.ra_bwd_pair(C.byref(p), a["out"], a["dtype"], *a["os"], a["dq"], *a["qs"], a["dk"], a["dv"], *a["ks"], a["ws"],
                               a["size"], None)

    need = lib.ra_bwd_pair_workspace(C.byref(_good_bwd()))
    assert need >= 12 * 2 * 64 and lib.ra_bwd_pair_workspace(None) == 0
    for kw, code in ((dict(out=None), -4), (dict(out=0x1008), -4), (dict(os=(64 * 128, 60, 128)), -4), (dict(dtype=3), -7),
                     (dict(dtype=_lib.RA_DTYPE_F16), -7), (dict(dq=None), -1), (dict(dk=None), -1), (dict(dv=None), -1),
                     (dict(dq=0x4004), -4), (dict(dv=0x6004), -4), (dict(ks=(64 * 128, 64, 126)), -4), (dict(ws=None), -4),
                     (dict(ws=0x7008), -4), (dict(size=need - 1), -2), (dict(mutate=lambda p: setattr(p, "lse", None)), -1),
                     (dict(mutate=lambda p: setattr(p.dout, "stride_h", 3)), -4), (dict(mutate=lambda p: setattr(p, "Lk", 0)), -2)):
        assert call(**kw) == code, kw
        assert lib.ra_last_error() != b""


def test_rows_beyond_a_32_bit_offset_are_refused_without_a_gpu(lib):
    # dK / dV reach -lse and -delta of a tile's 32 rows through one 32-bit byte offset, 4 (B H Lq + 31) at most; head dim 32 has no
    # kernel that does without.  32767 * 32769 = 2^30 - 1 rows are too many, 64 * 16777215 = 2^30 - 64 are not (refused later: no workspace)
    def call(H, Lq):
        p = _good_bwd()
        p.D, p.H, p.Lq = 32, H, Lq
        return lib.ra_bwd_whole(C.byref(p), 0x1000, _lib.RA_DTYPE_BF16, 64 * 128, 64, 128, _lib.RA_DTYPE_BF16, 0x4000, 64 * 128, 64, 128,
                                0x5000, 0x6000, 64 * 128, 64, 128, None, 0, None)

    assert call(32767, 32769) == _lib.RA_ERR_TOO_LARGE
    assert call(64, 16777215) == -4


def _rows(**kw):
    a = {**dict(src=0x1000, dst=0x2000, sd=_lib.RA_DTYPE_F32, dd=_lib.RA_DTYPE_BF16, d=96, to=128, B=1, L=4, H=2), **kw}
    return bytes(_lib.RaRows(a["src"], a["dst"], a["sd"], a["dd"], a["d"], a["to"], a["B"], a["L"], a["H"], 0, 192, 96, 0, 256, 128))


def test_convert_rejects_bad_arguments_without_a_gpu(lib):
    assert lib.ra_convert(None, 1, None) == -1
    for n in (0, -1, _lib.RA_MAX_CONVERT + 1):
        assert lib.ra_convert(_rows() * 5, n, None) == -2
    for kw, code in ((dict(src=0), -1), (dict(dst=0), -1), (dict(B=0), -2), (dict(L=-1), -2), (dict(H=0), -2), (dict(d=0), -2),
                     (dict(to=129), -3), (dict(d=256), -3), (dict(sd=3), -7), (dict(dd=-1), -7), (dict(src=0x1002), -4),
                     (dict(dst=0x2001), -4), (dict(B=65536), -8), (dict(L=1 << 26), -8), (dict(H=1 << 27), -8)):
        assert lib.ra_convert(_rows(**kw), 1, None) == code, kw
        assert lib.ra_convert(_rows() + _rows(**kw), 2, None) == code, kw  # every array is checked before anything is launched


def test_header_is_plain_c(tmp_path):
    """include/ring_attention_hip.h must compile as C99 on its own (no HIP, no C++)."""
    import shutil
    import subprocess
    gcc = shutil.which("gcc")
    if gcc is None:
        pytest.skip("no gcc")
    src = tmp_path / "hdr.c"
    src.write_text('#include "ring_attention_hip.h"\n#include <stddef.h>\n'
                   f"typedef char size_of_ra_rows[sizeof(ra_rows) == {C.sizeof(_lib.RaRows)} ? 1 : -1];\n"
                   "typedef char place_of_strides[offsetof(ra_rows, src_stride_b) == 48 ? 1 : -1];\n"
                   "int main(void) { ra_fwd_step_params p; (void)p; return RA_OK; }\n")
    res = subprocess.run([gcc, "-std=c99", "-Wall", "-Wextra", "-pedantic", "-Werror", "-fsyntax-only",
                          "-I", os.path.join(ROOT, "include"), str(src)], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr


def test_calls_are_checked_before_their_conversions_without_a_gpu(lib):
    # the conversions are in order (on a machine without a GPU their launch would fail as such); the call behind them is not
    fwd, bwd = _good_fwd(), _good_bwd()

    def forward(rows, n, size=1 << 30, lse=0x2000):
        return lib.ra_fwd_call(rows, n, bytes(fwd), 0x1000, 0, 64 * 256, 128, 256, lse, 0x3000, size, None)

    def backward(rows, n, size=1 << 30, dv=0x6000):
        return lib.ra_bwd_call(rows, n, bytes(bwd), 0x1000, 0, 64 * 128, 64, 128, 0, 0x4000, 64 * 128, 64, 128, 0x5000, dv, 64 * 128, 64, 128,
                               0x7000, size, None)

    assert forward(_rows(), 1, lse=None) == -1 and backward(_rows(), 1, dv=None) == -1 and backward(_rows(), 1, size=64) == -2
    for p, call in ((fwd, forward), (bwd, backward)):
        for n in (-1, _lib.RA_MAX_CONVERT + 1):
            assert call(_rows() * 5, n) == -2
        assert call(None, 1) == -1 and call(_rows(src=0x1002), 1) == -4
        p.D = 48
        assert call(_rows(), 1) == -3
        p.D, p.bias.flags = 64, 64
        assert call(_rows(), 1) == -5
    fwd.bias.flags, fwd.Lk = 0, 4096  # rows whose keys are shared
    assert forward(_rows(), 1, size=64) == -2
