"""Buffer ranges of operands whose rows start at any 2-byte address. Such kernels read whole dwords, so the
range that a bound launch gives them has to hold every element and end in the dword of the last one: one
dword more may lie past the end of the allocation. Checked on the host, on the argument blocks that bind_args
makes of dry plans, for both parities of the start and of the element count."""
import os
import shutil
import subprocess

import pytest

import example_matmul_metal4_amd as mtk

ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

DRIVER = r"""
#include "runtime.cpp"
// The kernels' view: dword-aligned base, range in bytes from there.
static int check(const char *what, uintptr_t p, uint64_t exact, uint32_t range) {
  const uint64_t base = p & ~(uintptr_t)3, end = p + exact;
  if (base + range >= end && base + range <= ((end + 3) & ~3ull)) return 0;
  printf("%s: start %% 4 = %d, %llu bytes, range %u ends %lld bytes past the operand\n", what, (int)(p & 3),
         (unsigned long long)exact, range, (long long)(base + range - end));
  return 1;
}
int main() {
  int bad = 0, seen = 0;
  for (int tb = 0; tb < 2; ++tb)
    for (int M : {3, 100, 1023, 1030})
      for (int N : {5, 300, 1023})
        for (int K : {7, 300, 1023})
          for (int pad : {0, 1, 2})
            for (int split : {0, 1, 3}) {
              mtk_gemm_desc d{};
              d.M = M, d.N = N, d.K = K, d.trans_b = tb, d.split_k = split, d.lda = K + pad, d.ldb = (tb ? K : N) + pad;
              mtk_plan *p = nullptr;
              if (mtk_gemm_plan(nullptr, &d, &p) != MTK_OK) return printf("no plan\n"), 1;
              if (p->align_a == 2)
                for (uintptr_t oa : {0, 2})
                  for (uintptr_t ob : {0, 2}) {
                    mtk_gemm_args g{};
                    g.A = (void *)(0x10000 + oa), g.B = (void *)(0x20000 + ob), g.C = (void *)0x30000, g.workspace = (void *)0x40000;
                    std::vector<Launch> ls;
                    if (bind_args(p, &g, ls) != MTK_OK) return printf("bind: %s\n", mtk_last_error()), 1;
                    const mtk_tile_args &a = args_of<mtk_tile_args>(ls[0]);
                    bad += check("A", (uintptr_t)g.A, 2ull * ((uint64_t)(M - 1) * d.lda + K), a.a_bytes);
                    bad += check("B", (uintptr_t)g.B, 2ull * ((uint64_t)((tb ? N : K) - 1) * d.ldb + (tb ? K : N)), a.b_bytes);
                    ++seen;
                  }
              mtk_plan_destroy(p);
            }
  for (int O : {5, 33, 65})  // quarter tiles with output channels of odd count
    for (uintptr_t ox : {0, 2})
      for (uintptr_t ow : {0, 2}) {
        mtk_conv_desc d{};
        d.rank = 2, d.N = 1, d.D = 1, d.H = 30, d.W = 13, d.C = 24, d.O = O, d.KD = 1, d.KH = d.KW = 3;
        d.stride_d = d.stride_h = d.stride_w = d.dil_d = d.dil_h = d.dil_w = 1;
        mtk_plan *p = nullptr;
        if (mtk_conv_plan(nullptr, &d, &p) != MTK_OK) return printf("no plan\n"), 1;
        mtk_conv_args c{};
        c.x = (void *)(0x10000 + ox), c.w = (void *)(0x20000 + ow), c.y = (void *)0x30000;
        std::vector<Launch> ls;
        if (bind_args(p, &c, ls) != MTK_OK) return printf("bind: %s\n", mtk_last_error()), 1;
        const mtk_tile_args &a = args_of<mtk_tile_args>(ls[0]);
        if (ls[0].name.find("_v1q") == std::string::npos) return printf("%s\n", ls[0].name.c_str()), 1;
        bad += check("x", (uintptr_t)c.x, 2ull * 30 * 13 * 24, a.a_bytes);
        bad += check("w", (uintptr_t)c.w, 2ull * 9 * 24 * O, a.b_bytes);
        mtk_plan_destroy(p);
        ++seen;
      }
  printf("%d launches, %d wrong ranges\n", seen, bad);
  return bad || seen < 100;
}
"""


def test_ranges_end_in_the_last_elements_dword(tmp_path):
    scratch_obj = os.path.join(mtk.LIB_DIR, "scratch.o")
    if shutil.which("g++") is None or not os.path.exists(scratch_obj):
        pytest.skip("needs g++ and a built library (python -m example_matmul_metal4_amd.build)")
    src, exe = tmp_path / "ranges.cpp", tmp_path / "ranges"
    src.write_text(DRIVER)
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM}/include",
                    f"-I{os.path.join(mtk.PKG, 'csrc')}", str(src), scratch_obj, f"-L{ROCM}/lib", "-lamdhip64",
                    f"-Wl,-rpath,{ROCM}/lib", "-ldl", "-o", str(exe)], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, (r.stdout + r.stderr)[-3000:]
