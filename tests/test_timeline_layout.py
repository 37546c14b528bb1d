"""The workspace layout of the profiling build (host code only, compiled here): the decode
chunks of a layer with I8 routed experts stamp their records also in a workspace that holds
no I8 GEMM scratch, so the record region has to end within the smallest one accepted."""
import subprocess
from pathlib import Path

from npu_amd import build as B

ROOT = Path(__file__).resolve().parents[1]

# gm_moe_ws_layout of capi.hip beside stand-ins for the sizes that other sources know
MAIN = r'''
#include <cstdio>
#include "kernels.h"
#include "timeline.h"
size_t gm_prefill_scratch_bytes(const gm_moe_layer*, int T) { return (size_t)T * 4096 + 40; }
size_t gm_pf8_scratch_bytes(const gm_moe_layer*, int T) { return (size_t)T * 70000 + 24; }
bool gm_pf8_ok(const gm_moe_layer*) { return true; }
int main() {
  gm_moe_layer L{};
  L.D = 2048; L.FF = L.FF_sh = 512; L.E = 16; L.k = 8;
  for (int T : {1, 8, 9, 101, 127, 4096}) {
    const GmMoeWs w = gm_moe_ws_layout(&L, T);
    std::printf("%d %zu %zu %zu %zu\n", T, w.tl, (size_t)GM_TL_BYTES, w.total_min, w.total);
  }
}
'''


def test_records_lie_in_the_smallest_workspace(tmp_path):
    src, exe = tmp_path / "layout.cpp", tmp_path / "layout"
    src.write_text(MAIN)
    inc = ["-I", str(ROOT / "include"), "-I", str(B.CSRC)]
    r = subprocess.run([B.hipcc(), "-x", "hip", "--offload-host-only", "-std=c++17", "-O1", "-DGM_TIMELINE=1", *inc,
                        "-ffunction-sections", "-Wl,--gc-sections", "-Wl,--unresolved-symbols=ignore-all",
                        str(B.CSRC / "capi.hip"), str(src), "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stderr[-2000:]
    rows = [[int(v) for v in line.split()] for line in out.stdout.splitlines()]
    assert [r[0] for r in rows] == [1, 8, 9, 101, 127, 4096]
    for T, tl, nbytes, least, total in rows:
        assert nbytes > 0 and tl + nbytes <= least <= total, T
        assert T > 8 or tl + nbytes == total            # where the timeline tool looks for them
