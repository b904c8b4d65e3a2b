"""Partial sums of attention plans that split the keys over workgroups, on the host: what any plan's kernels write fits
the region that a context has for a stream, and every kernel that a plan may run, with a region and without,
is in the built code objects."""
import glob
import os
import shutil
import subprocess

import pytest

import example_matmul_metal4_amd as mtk

ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

DRIVER = r"""
#include "runtime.cpp"
#include <random>
#include <set>
int main() {
  mtk_ctx ctx;
  ctx.prop.multiProcessorCount = 256;  // what dry plans are made for
  std::mt19937 rng(7);
  auto log = [&](int lo, int hi) { return (int)(lo * std::pow((double)hi / lo, std::uniform_real_distribution<>(0, 1)(rng))); };
  std::set<std::string> names;
  int split = 0;
  size_t most = 0;
  for (int n = 0; n < 200000; ++n) {
    mtk_attn_desc d{};
    const int groups[] = {1, 1, 2, 3, 4, 8, 16};
    d.B = log(1, 16), d.H_kv = log(1, 33), d.H = d.H_kv * groups[rng() % 7], d.S_kv = log(97, 40000), d.D = 8 * log(1, 33);
    d.S_q = rng() % 2 ? log(1, 70) : log(1, 2000), d.causal = rng() % 2, d.dtype = rng() % 2 ? MTK_F16 : MTK_BF16;
    mtk_plan *p = nullptr;
    if (mtk_attn_plan(nullptr, &d, &p) != MTK_OK) continue;
    for (auto *ls : {&p->launches, &p->plain})
      for (const Launch &l : *ls) names.insert(l.name);
    if (p->needs_part) {
      ++split;
      const mtk_attn_kargs &a = args_of<mtk_attn_kargs>(p->launches[0]), &c = args_of<mtk_attn_kargs>(p->launches[1]);
      const size_t rows = (size_t)d.B * d.H_kv * a.q_blocks * a.kv_splits * 32;
      const bool ok = a.part_ld >= d.D && rows * a.part_ld * 4 <= p->part_ml_at && p->part_ml_at + rows * 8 <= p->part_bytes &&
                      p->part_bytes <= ctx.part_capacity() && ctx.part_capacity() % 16 == 0 && p->part_ml_at % 8 == 0 &&
                      c.part_ld == a.part_ld && c.kv_splits == a.kv_splits && p->plain.size() == 1 &&
                      args_of<mtk_attn_kargs>(p->plain[0]).kv_splits == a.kv_splits;
      most = std::max(most, p->part_bytes);
      if (!ok) return printf("%s: %zu bytes\n", p->description.c_str(), p->part_bytes), 1;
    }
    mtk_plan_destroy(p);
  }
  for (auto &n : names) printf("%s\n", n.c_str());
  fprintf(stderr, "%d plans split, at most %zu of %zu bytes\n", split, most, ctx.part_capacity());
  return split < 1000;
}
"""


def test_partial_sums_fit_a_region(tmp_path):
    scratch_obj = os.path.join(mtk.LIB_DIR, "scratch.o")
    if shutil.which("g++") is None or not os.path.exists(scratch_obj):
        pytest.skip("needs g++ and a built library (python -m example_matmul_metal4_amd.build)")
    src, exe = tmp_path / "regions.cpp", tmp_path / "regions"
    src.write_text(DRIVER)
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM}/include",
                    f"-I{os.path.join(mtk.PKG, 'csrc')}", str(src), scratch_obj, f"-L{ROCM}/lib", "-lamdhip64",
                    f"-Wl,-rpath,{ROCM}/lib", "-ldl", "-o", str(exe)], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, (r.stdout + r.stderr)[-3000:]
    names = r.stdout.split()
    assert any("_seq_" in n for n in names) and any("combine" in n for n in names)
    built = b"".join(open(f, "rb").read() for f in glob.glob(os.path.join(mtk.LIB_DIR, "mtk_attention*.hsaco")))
    assert [n for n in names if n.encode() + b"\0" not in built] == []
