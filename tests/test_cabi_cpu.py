"""Host-side checks that need no GPU: the shared library loads, exports every symbol the header
declares, agrees with the Python binding on the struct layout, and fa_validate returns the
documented code for each malformed argument.  The operator's Python layer raises the same
AssertionErrors as the reference (flash_triton.py:510-530) before touching the GPU."""
import ctypes
import re
from pathlib import Path

import pytest
import torch

from flash_mi355 import _cabi, attention, SCORE_FUNC_MODE1_DOC

ROOT = Path(__file__).resolve().parent.parent
HEADER = (ROOT / "include" / "flash_mi355.h").read_text()


def _declared_functions():
    body = HEADER.split('extern "C" {')[1]
    return sorted(set(re.findall(r"^\s*(?:const\s+)?[a-z_0-9]+\*?\s+(fa_[a-z_0-9]+)\s*\(", body, re.M)))


def test_library_exports_every_declared_symbol():
    L = _cabi.lib()
    names = _declared_functions()
    assert set(names) == set(_cabi.EXPORTS), (names, _cabi.EXPORTS)
    for n in names:
        assert getattr(L, n) is not None


def test_clock_stamp_build_is_a_library_of_its_own():
    """bench.py --wg-trace loads libflash_mi355_trace.so: every entry point of the header plus
    fa_trace_read.  The product library carries no trace export."""
    from flash_mi355.build import TRACE_LIB_PATH
    assert TRACE_LIB_PATH.exists(), "python -m flash_mi355.build builds it next to the product library"
    T = ctypes.CDLL(str(TRACE_LIB_PATH))
    for n in _declared_functions() + ["fa_trace_read"]:
        assert getattr(T, n) is not None
    T.fa_version.restype = ctypes.c_int
    assert T.fa_version() == _cabi.FA_ABI_VERSION
    with pytest.raises(AttributeError):
        _cabi.lib().fa_trace_read


def test_struct_layout_and_version():
    L = _cabi.lib()
    assert L.fa_version() == _cabi.FA_ABI_VERSION == int(re.search(r"#define FA_ABI_VERSION (\d+)", HEADER).group(1))
    assert L.fa_params_size() == ctypes.sizeof(_cabi.FaParams)
    for code in range(0, -11, -1):
        assert L.fa_error_string(code)


def _good_params(buf):
    p = _cabi.FaParams()
    base = (ctypes.addressof(buf) + 255) & ~255
    for f in ("q", "k", "v", "o", "lse", "dout", "dq", "dk", "dv", "delta"):
        setattr(p, f, base)
    p.B, p.H, p.Hk, p.M, p.N, p.D = 1, 4, 2, 128, 256, 64
    for f in ("q_stride", "o_stride", "do_stride", "dq_stride"):
        arr = getattr(p, f); arr[0], arr[1], arr[2], arr[3] = 4 * 128 * 64, 128 * 64, 64, 1
    for f in ("k_stride", "v_stride", "dk_stride", "dv_stride"):
        arr = getattr(p, f); arr[0], arr[1], arr[2], arr[3] = 4 * 256 * 64, 256 * 64, 64, 1
    p.causal, p.score_mode, p.dtype, p.sm_scale = 1, 0, _cabi.FA_DTYPE_BF16, 0.125
    return p


def test_validate_codes():
    L = _cabi.lib()
    buf = ctypes.create_string_buffer(4096)
    v = lambda p, stage=1: L.fa_validate(ctypes.byref(p), stage)
    assert v(_good_params(buf)) == 0
    assert L.fa_validate(None, 0) == -1
    p = _good_params(buf); p.D = 48; assert v(p) == -2           # flash_triton.py:512
    p = _good_params(buf); p.D = 256; assert v(p) == -2
    p = _good_params(buf); p.dtype = 5; assert v(p) == -3
    p = _good_params(buf); p.H = 3; assert v(p) == -4             # H % Hk, flash_triton.py:518
    p = _good_params(buf); p.M, p.N = 256, 128; assert v(p) == -4  # causal needs N >= M, flash_triton.py:520
    p = _good_params(buf); p.M, p.N, p.causal = 256, 128, 0; assert v(p) == 0
    p = _good_params(buf); p.B = 0; assert v(p) == -4
    p = _good_params(buf); p.q += 8; assert v(p) == -5
    p = _good_params(buf); p.q_stride[2] = 68; assert v(p) == -5
    p = _good_params(buf); p.k_stride[3] = 2; assert v(p) == -6
    p = _good_params(buf); p.score_mode = 3; assert v(p) == -7
    p = _good_params(buf); p.score_mode = 1; assert v(p) == -7     # doc mode without ids
    p = _good_params(buf); p.score_mode = 1; p.eq = p.ek = p.q; assert v(p) == -8   # no workspace
    p = _good_params(buf); p.dout = None; assert v(p, 1) == -1 and v(p, 0) == 0
    p = _good_params(buf); p.flags = 2; assert v(p) == -7
    # the diagnostic flag of the dk/dv pair wait is honoured by fa_bwd_dkdv's stage alone
    p = _good_params(buf); p.flags = _cabi.FA_FLAG_DEBUG_NO_PAIR_WAIT
    assert v(p, 3) == 0 and v(p, 0) == -7 and v(p, 1) == -7 and v(p, 2) == -7
    p = _good_params(buf); p.dout = None; assert v(p, 3) == -1
    # per-row causal positions: only with causal + ids, not with a prefix; they lift the N >= M rule
    p = _good_params(buf); p.qpos = p.q; assert v(p) == -7           # no ids
    p = _good_params(buf); p.qpos = p.q; p.score_mode = 1; p.eq = p.ek = p.q; p.causal = 0; assert v(p, 2) == -7
    p = _good_params(buf); p.qpos = p.q; p.score_mode = 1; p.eq = p.ek = p.q; p.prefix = 4; assert v(p, 2) == -7
    p = _good_params(buf); p.qpos = p.q; p.score_mode = 1; p.eq = p.ek = p.q; p.M, p.N = 256, 128; assert v(p, 2) == -8   # past the shape check: no workspace
    p = _good_params(buf); p.flags = _cabi.FA_FLAG_DQ_DELTA; assert v(p) == 0 and v(p, 1) == 0
    p = _good_params(buf); p.flags = _cabi.FA_FLAG_DQ_DELTA; p.dtype = _cabi.FA_DTYPE_FP32; assert v(p, 1) == 0
    # block mask: eq carries the byte map, no workspace, no ek; rows of the map at least ceil(N/64) apart
    p = _good_params(buf); p.score_mode = _cabi.FA_SCORE_MODE2_BLOCK; assert v(p) == -7
    p = _good_params(buf); p.score_mode = _cabi.FA_SCORE_MODE2_BLOCK; p.eq = p.q; p.eq_stride[2] = (p.N + 63) // 64
    assert v(p) == 0 and L.fa_workspace_bytes(ctypes.byref(p)) == 0
    p.eq_stride[2] -= 1; assert v(p) == -6
    p.eq_stride[2] += 1; p.dtype = _cabi.FA_DTYPE_FP32; assert v(p) == 0
    # sliding window / prefix: causal only, not both, not negative
    p = _good_params(buf); p.window = 64; assert v(p) == 0
    p = _good_params(buf); p.prefix = 64; assert v(p) == 0
    p = _good_params(buf); p.window = 64; p.prefix = 8; assert v(p) == -7
    p = _good_params(buf); p.window = -1; assert v(p) == -7
    p = _good_params(buf); p.M, p.N, p.causal, p.window = 256, 128, 0, 16; assert v(p) == -7
    # fp32 tensors are accepted; their strides must be multiples of 16 bytes = 4 elements
    p = _good_params(buf); p.dtype = _cabi.FA_DTYPE_FP32; assert v(p) == 0
    p = _good_params(buf); p.dtype = _cabi.FA_DTYPE_FP32; p.q_stride[2] = 68; assert v(p) == 0
    p = _good_params(buf); p.dtype = _cabi.FA_DTYPE_FP32; p.q_stride[2] = 66; assert v(p) == -5


def test_workspace_size():
    L = _cabi.lib()
    buf = ctypes.create_string_buffer(4096)
    p = _good_params(buf)
    assert L.fa_workspace_bytes(ctypes.byref(p)) == 0
    p.score_mode = 1
    p.eq_stride[0], p.eq_stride[1], p.eq_stride[2] = 128, 0, 1       # ids shared by the heads
    p.ek_stride[0], p.ek_stride[1], p.ek_stride[2] = 4 * 256, 256, 1   # per head
    r256 = lambda x: (x + 255) // 256 * 256
    Pp = 256 + 256
    want = (r256(128 * 4) + r256(4 * 256 * 4) + 3 * r256(Pp * 4) + r256(4) + r256(32) + r256(Pp // 64 * 32)
            + r256(4 * 4 * 32))
    assert L.fa_workspace_bytes(ctypes.byref(p)) == want   # 4 key tiles of 64: no key range is ever split
    assert L.fa_workspace_plan_bytes(ctypes.byref(p)) == want   # ... so all of it is plan
    # from 32 key tiles on, scratch for split global-row tiles: arrival counters, (max, sum) pairs, fp32
    # partial tiles; chunks = clamp(key tiles / 32, 2, 4) (finer when the launch is short of workgroups),
    # splittable tiles = min(128 MiB / footprint, 64), at most ceil(M / 128) + 1
    p.N = 2048
    p.ek_stride[0], p.ek_stride[1] = 4 * 2048, 2048
    chunks, tiles = 2, 2   # 32 key tiles -> 2 chunks of 16; M = 128 rows -> 2 tiles
    assert p.M == 128 and (128 << 20) // (1 * 4 * chunks * 128 * (p.D + 2) * 4) >= 64
    want = (r256(128 * 4) + r256(4 * 2048 * 4) + 3 * r256(Pp * 4) + r256(4) + r256(32) + r256(Pp // 64 * 32)
            + r256(4 * 32 * 32)
            + r256(4 * tiles * 4) + r256(4 * tiles * chunks * 128 * 2 * 4) + r256(4 * tiles * chunks * 128 * p.D * 4))
    assert L.fa_workspace_bytes(ctypes.byref(p)) == want
    # the plan proper (what has to survive from forward to backward) ends after the counters
    scratch = r256(4 * tiles * chunks * 128 * 2 * 4) + r256(4 * tiles * chunks * 128 * p.D * 4)
    assert L.fa_workspace_plan_bytes(ctypes.byref(p)) == want - scratch


@pytest.mark.parametrize("M,N,low", [(511, 4096, False), (512, 4096, True), (2000, 16384, True), (12200, 12200, True), (12400, 12400, False), (33000, 33000, False)])
def test_workspace_does_not_depend_on_qpos(M, N, low):
    """Rows with positions of their own take query tiles of 128 rows where others take 64; the arrival counters are as many for both."""
    L = _cabi.lib()
    buf = ctypes.create_string_buffer(4096)
    p = _good_params(buf)
    p.M, p.N, p.score_mode = M, N, 1
    p.eq_stride[0], p.eq_stride[2], p.ek_stride[0], p.ek_stride[2] = M, 1, N, 1
    want = [f(ctypes.byref(p)) for f in (L.fa_workspace_bytes, L.fa_workspace_plan_bytes)]
    p.qpos = p.q
    assert [f(ctypes.byref(p)) for f in (L.fa_workspace_bytes, L.fa_workspace_plan_bytes)] == want
    r256 = lambda x: (x + 255) // 256 * 256
    Pp, Mp, Np = r256(M) + 256, -(-M // 64) * 64, -(-N // 64) * 64
    ids = r256(Mp * 4) + r256(Np * 4) + 3 * r256(Pp * 4) + r256(-(-Mp // 1024) * 4) + r256(32) + r256(Pp // 64 * 32) + r256(Np // 64 * 32)
    tiles = min(64, -(-M // 128) + 1)
    assert want[1] - ids == r256(p.H * tiles * (2 if low else 1) * 4)


@pytest.mark.parametrize("M,N", [(1, 16384), (100, 9000), (3, 300), (2000, 16384), (4096, 4096)])
def test_a_window_past_every_key_is_no_window(M, N):
    """Window sizes up to the largest int (callers that mean "none") shape the launch like window = 0: the form and the
    chunks of the key range, seen in the workspace they ask for."""
    L = _cabi.lib()
    buf = ctypes.create_string_buffer(4096)
    p = _good_params(buf)
    p.M, p.N, p.flags = M, N, _cabi.FA_FLAG_SPLIT_KEYS
    want = L.fa_workspace_bytes(ctypes.byref(p))
    assert (want > 0) == (N > 8000)
    for window in (N, N + M, (1 << 30) - 1, 1 << 30, (1 << 31) - 1 - M, (1 << 31) - M, (1 << 31) - 1):
        p.window = window
        assert L.fa_workspace_bytes(ctypes.byref(p)) == want, window
    p.window = 64   # a real one leaves short ranges, which are not cut
    assert M != 1 or L.fa_workspace_bytes(ctypes.byref(p)) == 0


def _packed_params(buf, nseq, M, N, H, Hk, D):
    p = _good_params(buf)
    p.score_mode, p.nseq, p.eq, p.ek = _cabi.FA_SCORE_MODE3_PACKED, nseq, p.k, p.k
    p.B, p.M, p.N, p.H, p.Hk, p.D = 1, M, N, H, Hk, D
    return p


def test_packed_rows_stay_inside_an_int(tmp_path):
    """Heads share tiles only while the packed rows, up to the end of the last tile, can be counted in int; the launch shape
    is compiled for the host from the header the launches use."""
    import os
    import subprocess
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    csrc = ROOT / "triton-flash-attention-with-flexible-masks_amd" / "csrc"
    src = tmp_path / "shape.hip"
    src.write_text(r'''
#include <cstdio>
#include "fa_common.h"
int main() {
  const int rows[][3] = {{1 << 26, 32, 1}, {1 << 26, 31, 1}, {1 << 26, 64, 2}, {(1 << 26) - 9, 32, 1}, {(1 << 26) - 4, 32, 1}, {1 << 26, 128, 8}, {333, 32, 8}, {1 << 26, 16, 16}};
  for (const auto& r : rows)
    for (int mode : {FA_SCORE_MODE0_NOPE, FA_SCORE_MODE3_PACKED}) {
      fa_params p = {};
      p.B = 1; p.M = r[0]; p.N = 1 << 20; p.H = r[1]; p.Hk = r[2]; p.D = 16; p.causal = 0; p.dtype = FA_DTYPE_BF16; p.score_mode = mode; p.nseq = 3;
      const fa::FwdCfg c = fa::fwd_config(&p);
      const long long last = ((long long)r[0] * c.pack + c.bm - 1) / c.bm * c.bm;
      printf("%d %d %d\n", r[1] / r[2], c.pack, last <= 0x7fffffffLL && (mode == FA_SCORE_MODE3_PACKED || (long long)c.tiles * c.bm == last));
    }
}
''')
    exe = tmp_path / "shape"
    subprocess.run([hipcc, "--offload-host-only", "-std=c++17", "-O1", f"-I{csrc}", str(src), "-o", str(exe)], check=True, capture_output=True)
    out = [tuple(map(int, l.split())) for l in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.splitlines()]
    assert len(out) == 16 and all(ok for _, _, ok in out), out
    assert [pack for _, pack, _ in out[::2]] == [1, 31, 1, 32, 1, 16, 4, 1] == [pack for _, pack, _ in out[1::2]], out


def test_gpu_cases_reach_the_query_tiles_they_are_written_for(tmp_path):
    """Tiles of 64 or 128 rows with ids, under a block map and under a causal mask alone, by the header the launches use."""
    import os
    import subprocess
    from tests import test_gpu_launch_forms as F
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    csrc = ROOT / "triton-flash-attention-with-flexible-masks_amd" / "csrc"
    calls = [f"fa::split_config({c[0] * c[10].get('copies', 1)}, {c[1]}, {c[3]}, {c[4]}, {c[5]}, {int('qpos' in c[10])}).rows" for c in F.LOW_TILE_CASES]
    calls += [f"fa::block_rows({c[0]}, {c[1]}, {c[3]}, {c[5]})" for c in F.LOW_BLOCK_CASES]
    calls += [f"dq_block(1, {c[0]}, {c[2]}, {c[3]}, 128)" for c in F.LONG_BLOCK_CASES]
    src = tmp_path / "rows.hip"
    calls += [f"causal({c[0] * c[8]}, {c[1]}, {c[2]}, {c[3]}, {c[4]}, {c[5]}, {c[7]}, {sum(c[11:])})" for c in F.LOW_CAUSAL_CASES]
    src.write_text('''#include <cstdio>
#include "fa_common.h"
static int causal(int B, int H, int Hk, int M, int N, int D, int prefix, int window) {
  fa_params p = {};
  p.B = B; p.H = H; p.Hk = Hk; p.M = M; p.N = N; p.D = D; p.prefix = prefix; p.window = window; p.causal = 1; p.dtype = FA_DTYPE_BF16; p.flags = FA_FLAG_SPLIT_KEYS;
  const fa::FwdCfg f = fa::fwd_config(&p), b = fa::fwd_config(&p, false);
  return !f.dec && f.split == 1 && b.split == 1 ? 1000 * f.bm + b.bm : 0;
}
static int dq_block(int B, int H, int M, int N, int D) {
  fa_params p = {};
  p.B = B; p.H = p.Hk = H; p.M = M; p.N = N; p.D = D; p.score_mode = FA_SCORE_MODE2_BLOCK; p.dtype = FA_DTYPE_BF16;
  return fa::fwd_config(&p, false).bm;
}
int main() { for (int r : {''' + ", ".join(calls) + '''}) printf("%d\\n", r); }
''')
    exe = tmp_path / "rows"
    subprocess.run([hipcc, "--offload-host-only", "-std=c++17", "-O1", f"-I{csrc}", str(src), "-o", str(exe)], check=True, capture_output=True)
    got = list(map(int, subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()))
    assert got == [c[9] for c in F.LOW_TILE_CASES] + [c[11] for c in F.LOW_BLOCK_CASES] + [c[5] for c in F.LONG_BLOCK_CASES] + \
        [1000 * c[9] + c[10] for c in F.LOW_CAUSAL_CASES]


def test_64_row_tiles_leave_the_static_forward_its_sizes(tmp_path):
    """fa_fwd_static takes what fits FA_STATIC_WS_BYTES with one arrival counter to 128 rows, whatever the tiles: its largest key ranges by the sizes of the
    layout's parts, at each one below and above (with ids, with positions as well)."""
    import os
    import subprocess
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    csrc = ROOT / "triton-flash-attention-with-flexible-masks_amd" / "csrc"
    cases = [(1, 1, 4096, 64), (1, 1, 8192, 128), (1, 2, 2000, 64), (1, 1, 700, 128), (2, 8, 3000, 64), (3, 32, 512, 64), (1, 1, 48000, 64), (1, 1, 300, 64)]
    src = tmp_path / "static.hip"
    src.write_text('''#include <cstdio>
#include "fa_common.h"
static bool fits(int B, int H, int M, int D, int N, bool own) {
  fa_params p = {};
  p.B = B; p.H = p.Hk = H; p.M = M; p.N = N; p.D = D; p.score_mode = FA_SCORE_MODE1_DOC;
  if (own) p.qpos = &N;
  const fa::WsLayout w = fa::ws_layout(&p, uint64_t(24) << 20);
  return fa::fits_static(w) && w.total <= FA_STATIC_WS_BYTES + fa::kStaticMargin;
}
int main(int c, char** v) {
  const int cases[][4] = {''' + ", ".join("{%d, %d, %d, %d}" % x for x in cases) + '''};
  for (auto& x : cases) for (bool own : {false, true}) {
    int lo = 1 << 14, hi = 1 << 24;
    while (hi - lo > 1) { const int m = lo + (hi - lo) / 2; (fits(x[0], x[1], x[2], x[3], m, own) ? lo : hi) = m; }
    fa_params p = {};
    p.B = x[0]; p.H = p.Hk = x[1]; p.M = x[2]; p.N = lo; p.D = x[3]; p.score_mode = FA_SCORE_MODE1_DOC;
    const fa::SplitCfg s = fa::split_config(p.B, p.H, p.M, p.N, p.D, own, uint64_t(24) << 20);
    printf("%d %d %d %d\\n", lo, s.k, s.tiles * s.rows / 128, s.rows);
  }
}
''')
    exe = tmp_path / "static"
    subprocess.run([hipcc, "--offload-host-only", "-std=c++17", "-O1", f"-I{csrc}", str(src), "-o", str(exe)], check=True, capture_output=True)
    got = [tuple(map(int, l.split())) for l in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.splitlines()]
    r256 = lambda x: (x + 255) // 256 * 256

    def total(B, H, M, D, N, k, tiles):
        Mp, Np, Pp = -(-M // 64) * 64, -(-N // 64) * 64, -(-M // 256) * 256 + 256
        plan = r256(B * Mp * 4) + r256(B * Np * 4) + 3 * r256(B * Pp * 4) + r256(B * -(-Mp // 1024) * 4) + r256(B * 32) + r256(B * Pp // 64 * 32) + r256(B * Np // 64 * 32)
        return plan + r256(B * H * tiles * 4) + r256(B * H * tiles * k * 128 * 2 * 4) + r256(B * H * tiles * k * 128 * D * 4)

    for i, (N, k, tiles, _) in enumerate(got):
        B, H, M, D = cases[i // 2]
        assert total(B, H, M, D, N, k, tiles) <= 32 << 20 < total(B, H, M, D, N + 1, k, tiles), (cases[i // 2], N)
    assert {r for _, _, _, r in got} == {64, 128} and all(got[i][0] == got[i + 1][0] for i in range(0, len(got), 2))


@pytest.mark.parametrize("nseq,M,N,H,Hk,D,bm", [
    (600, 15000, 15000, 8, 8, 128, 64),      # many short sequences: not the form with one workgroup to a CU
    (600, 15000, 15000, 32, 32, 64, 64),
    (1001, 5096, 350000, 32, 8, 128, 64),    # 1000 decoding sequences and a prompt
    (64, 512, 64 * 500, 32, 8, 128, 64),
    (64, 512, 64 * 1024, 32, 8, 128, 32),     # long key ranges
    (64, 512, 64 * 2048, 16, 16, 64, 64),
    (64, 512, 64 * 4096, 16, 16, 64, 32),
    (16, 256, 16 * 100, 8, 8, 128, 32),      # few tiles
    (17, 512, 17 * 100, 8, 8, 128, 64),
    (24, 15000, 15000, 32, 8, 128, 128),
])
def test_tile_height_of_packed_sequences(nseq, M, N, H, Hk, D, bm):
    """The tables are laid out for the tile height the totals ask for; the decode form (32 rows) is for few tiles or
    long key ranges."""
    L = _cabi.lib()
    buf = ctypes.create_string_buffer(4096)
    p = _packed_params(buf, nseq, M, N, H, Hk, D)
    r256 = lambda x: (x + 255) // 256 * 256
    spare = 448 // Hk + 1
    plan = lambda b: (256 + r256((M * (H // Hk) // b + nseq + 1 + spare) * 64) + r256((N // (64 if D > 64 else 128) + nseq + 1) * 64)
                      + r256(spare * Hk * 4))
    assert [b for b in (32, 64, 128) if plan(b) == L.fa_workspace_plan_bytes(ctypes.byref(p))] == [bm]


def test_static_forward_never_takes_a_workspace_that_nobody_planned():
    """fa_fwd_static ignores p->workspace: what would read tables or counters out of it is refused (packed sequences) or
    left out (split key ranges).  No operand is set, so the call ends at the checks, with a GPU or without."""
    L = _cabi.lib()
    buf = ctypes.create_string_buffer(4096)
    p = _good_params(buf)
    p.q = None
    p.workspace, p.workspace_bytes = 256 * 1024, 1 << 40    # a filled struct that was used before
    assert L.fa_fwd_static(ctypes.byref(p), None) == -1
    p.score_mode, p.nseq, p.eq, p.ek, p.B = _cabi.FA_SCORE_MODE3_PACKED, 2, p.k, p.k, 1
    assert L.fa_fwd_static(ctypes.byref(p), None) == -7
    # one row against a long key range is split when the flag is set and a workspace is there
    p = _good_params(buf)
    p.q, p.M, p.N = None, 1, 16384
    p.flags = _cabi.FA_FLAG_SPLIT_KEYS
    assert L.fa_workspace_bytes(ctypes.byref(p)) > 0 and L.fa_validate(ctypes.byref(p), 0) == -8
    assert L.fa_fwd_static(ctypes.byref(p), None) == -1     # no workspace asked for: the flag is left out


def test_static_forward_leaves_the_callers_split_scratch_alone():
    """The scratch of the split key ranges lies in the library's array: a split_scratch left over in the struct (here a
    misaligned one) is neither used nor looked at.  No operand is set, so the call ends at the checks."""
    L = _cabi.lib()
    buf = ctypes.create_string_buffer(4096)
    p = _good_params(buf)
    p.score_mode, p.eq, p.ek, p.N, p.q = 1, p.k, p.k, 4096, None
    p.split_scratch, p.split_scratch_bytes = 256 * 1024 + 64, 64
    assert L.fa_workspace_scratch_bytes(ctypes.byref(p)) > 64
    assert L.fa_fwd_static(ctypes.byref(p), None) == -1


def test_python_layer_asserts_like_the_reference():
    q = torch.zeros(1, 4, 8, 64, dtype=torch.bfloat16)
    k = torch.zeros(1, 2, 16, 64, dtype=torch.bfloat16)
    e_q = torch.zeros(1, 4, 8, dtype=torch.int32)
    with pytest.raises(AssertionError):
        attention(q, k, torch.zeros(1, 2, 16, 32, dtype=torch.bfloat16))          # feature sizes differ
    with pytest.raises(AssertionError):
        attention(torch.zeros(1, 4, 8, 48), torch.zeros(1, 2, 16, 48), torch.zeros(1, 2, 16, 48))   # D not in {16,32,64,128}
    with pytest.raises(AssertionError):
        attention(q, k, torch.zeros(1, 1, 16, 64, dtype=torch.bfloat16))          # kv head counts differ
    with pytest.raises(AssertionError):
        attention(torch.zeros(1, 3, 8, 64), k, k)                                   # H % Hk
    with pytest.raises(AssertionError):
        attention(torch.zeros(1, 4, 32, 64, dtype=torch.bfloat16), k, k, causal=True)   # causal with N < M
    with pytest.raises(AssertionError):
        attention(q, k, k, eq=e_q)                                                  # eq without ek
    with pytest.raises(AssertionError):
        attention(q, k, k, score_func_mode=SCORE_FUNC_MODE1_DOC)                    # doc mode without ids
    with pytest.raises(AssertionError):
        attention(q, k, k)                                                          # CPU tensors: no CPU fallback


def test_the_packed_mode_is_not_a_score_func_mode():
    """Mode 3 is how attention_varlen hands packed sequences on; given as score_func_mode (with vectors that would pass
    for cumulative lengths) it is refused like any unknown mode, before the device of the operands is looked at."""
    from flash_mi355 import api
    q = torch.zeros(1, 4, 8, 64, dtype=torch.bfloat16)
    cu = torch.tensor([0, 3, 8], dtype=torch.int32)
    for f in (attention, api.attention_with_lse):
        for mode in (3, 4, -1):
            with pytest.raises(AssertionError, match="unknown score_func_mode"):
                f(q, q, q, True, None, cu, cu, mode)
    for cls in (api.FlashAttention, api.FlashAttentionWithLse):
        with pytest.raises(AssertionError, match="unknown score_func_mode"):
            cls.apply(q, q, q, True, None, cu, cu, 3)
    with pytest.raises(AssertionError, match="KV length"):   # ... and does not lift the rule on lengths
        attention(q, q[:, :, :4], q[:, :, :4], True, None, cu, cu, 3)
    with pytest.raises(AssertionError, match="GPU only"):    # the packed path's own calls pass the check
        api.attention_varlen(q[0], q[0], q[0], cu)


def test_which_packed_batches_go_through_the_document_mask():
    from flash_mi355 import api
    f = api._host().varlen_as_documents
    assert f(20000, 20000, 1000, 8, 8, 128, True)          # 20 tokens on average, 8000 tiles
    assert not f(20000, 20000, 500, 8, 8, 128, True)       # 40 tokens on average
    assert not f(8000, 8000, 500, 8, 8, 128, True)         # 16, but 4000 tiles only
    assert f(8000, 8000, 500, 8, 8, 128, True) == f(8000, 8000, 1000, 8, 8, 64, True) == False
    assert f(8000, 8000, 512, 8, 8, 128, True) and f(8000, 8000, 1024, 8, 8, 64, True)
    assert f(20000, 20000, 1200, 32, 8, 128, True) and not f(20000, 20000, 1000, 32, 8, 128, True)   # groups of four fill tiles sooner
    assert not f(20000, 20000, 1000, 8, 8, 128, False) and f(20000, 20000, 3000, 8, 8, 128, False)   # positions cost more
    assert not f(3000, 90000, 3000, 32, 8, 128, False)     # queries on a cache of keys
    assert not f(3000, 3000, 3000, 8, 0, 128, True)        # (no key heads: refused later)
    assert not f(1 << 31, 1 << 31, 1 << 24, 8, 8, 128, True) and f(1 << 31, 1 << 31, 1 << 28, 8, 8, 128, True)


def test_operands_on_another_device_are_refused():
    """Ids, k, v or dO that do not live on q's device are refused with an AssertionError before any
    pointer reaches a kernel (checked on the helper itself: no GPU is needed to compare devices)."""
    from flash_mi355 import api
    q = torch.zeros(1, 1, 8, 16, device="meta")
    api._check_same_device(q, k=torch.zeros(2, device="meta"), eq=None)
    with pytest.raises(AssertionError, match="eq is on cpu"):
        api._check_same_device(q, eq=torch.zeros(1, 1, 8, dtype=torch.int32))
    with pytest.raises(AssertionError, match="v is on cpu"):
        api._check_same_device(q, k=torch.zeros(2, device="meta"), v=torch.zeros(2))
    import inspect
    src = inspect.getsource(api._Impl.forward) + inspect.getsource(api._Impl.backward)
    assert src.count("_check_same_device(q, ") >= 3   # k/v, eq/ek in forward; dO in backward


def test_split_scratch_stays_inside_its_budget():
    """The scratch of the split key ranges is bounded whatever the batch: with many (batch, head) pairs
    fewer tiles per pair are splittable, down to none."""
    L = _cabi.lib()
    buf = ctypes.create_string_buffer(4096)
    budget = 128 << 20
    for (B, H, Lseq, D) in [(64, 32, 2048, 128), (32, 32, 4096, 128), (8, 32, 8192, 128), (1, 32, 16384, 128),
                            (4, 8, 65536, 64), (256, 64, 2048, 16), (1, 4, 131072, 128)]:
        p = _good_params(buf)
        p.B, p.H, p.Hk, p.M, p.N, p.D = B, H, H, Lseq, Lseq, D
        p.score_mode = 1
        p.eq_stride[0], p.eq_stride[1], p.eq_stride[2] = Lseq, 0, 1
        p.ek_stride[0], p.ek_stride[1], p.ek_stride[2] = Lseq, 0, 1
        total = L.fa_workspace_bytes(ctypes.byref(p))
        plan = L.fa_workspace_plan_bytes(ctypes.byref(p))
        assert 0 < plan <= total and total - plan <= budget + 512, (B, H, Lseq, D, total - plan)
        assert L.fa_workspace_scratch_bytes(ctypes.byref(p)) == total - plan
        # a workspace of the plan's size is enough once the scratch has a home of its own
        p.workspace, p.workspace_bytes = 256 * 1024, plan
        p.eq = p.ek = p.q
        assert L.fa_validate(ctypes.byref(p), 2) == (-8 if total > plan else 0)
        p.split_scratch, p.split_scratch_bytes = 512 * 1024, total - plan
        assert L.fa_validate(ctypes.byref(p), 2) == 0
        p.split_scratch += 64
        assert L.fa_validate(ctypes.byref(p), 2) == -5
        p.split_scratch -= 64
        if total > plan:
            p.split_scratch_bytes -= 1
            assert L.fa_validate(ctypes.byref(p), 2) == -8
            p.split_scratch_bytes += 1
        p.workspace_bytes = plan - 1
        assert L.fa_validate(ctypes.byref(p), 2) == -8
    # the headline shape still splits its global-row tiles
    p = _good_params(buf)
    p.B, p.H, p.Hk, p.M, p.N, p.D, p.score_mode = 1, 32, 32, 16384, 16384, 128, 1
    p.eq_stride[2] = p.ek_stride[2] = 1
    assert L.fa_workspace_bytes(ctypes.byref(p)) - L.fa_workspace_plan_bytes(ctypes.byref(p)) > (32 << 20)


def test_drop_in_module_name():
    import flash_triton
    import flash_mi355
    assert flash_triton.attention is flash_mi355.attention
    assert flash_triton.FlashAttention is flash_mi355.FlashAttention
    assert (flash_triton.SCORE_FUNC_MODE0_NOPE, flash_triton.SCORE_FUNC_MODE1_DOC) == (0, 1)
    import inspect
    sig = inspect.signature(flash_triton.attention)
    pos = [n for n, p in sig.parameters.items() if p.kind == p.POSITIONAL_OR_KEYWORD]
    assert pos == ["q", "k", "v", "causal", "sm_scale", "eq", "ek", "score_func_mode"]   # flash_triton.py:640
    extra = {n: p for n, p in sig.parameters.items() if n not in pos}
    assert all(p.kind == p.KEYWORD_ONLY and p.default in (0, None) for p in extra.values())   # additions stay out of the way, default off
    assert [sig.parameters[n].default for n in pos][3:] == [False, None, None, None, 0]


def test_header_is_plain_c_and_matches_the_binding(tmp_path):
    """include/flash_mi355.h compiles as C (no C++ or HIP types in the boundary), a C program linked
    against the library sees the same struct size as the ctypes mirror, and validation works from C."""
    import shutil
    import subprocess
    if shutil.which("gcc") is None:
        pytest.skip("no gcc")
    src = tmp_path / "abi.c"
    src.write_text(r'''
#include <stdio.h>
#include <string.h>
#include "flash_mi355.h"
int main(void) {
  fa_params p;
  memset(&p, 0, sizeof p);
  printf("%d %llu %llu %d %s\n", fa_version(), (unsigned long long)fa_params_size(), (unsigned long long)sizeof(fa_params),
         fa_validate(&p, 0), fa_error_string(fa_validate(&p, 0)));
  return 0;
}
''')
    exe = tmp_path / "abi"
    lib_dir = _cabi.LIB_PATH.parent
    inc = Path(__file__).resolve().parent.parent / "include"
    subprocess.run(["gcc", "-std=c99", "-Wall", "-Werror", f"-I{inc}", str(src), "-o", str(exe), f"-L{lib_dir}",
                    "-lflash_mi355", f"-Wl,-rpath,{lib_dir}"], check=True, capture_output=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split(None, 4)
    assert int(out[0]) == _cabi.FA_ABI_VERSION
    assert int(out[1]) == int(out[2]) == ctypes.sizeof(_cabi.FaParams)
    assert int(out[3]) == -2 and "head dimension" in out[4]      # D = 0 is the first thing a zeroed struct fails
