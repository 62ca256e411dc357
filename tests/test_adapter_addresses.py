"""The kernel_interface adapter publishes the addresses of p, u, r, w and sd
anew after every call that can exchange a field's buffers.  The adapter is
linked to a stand-in for the library whose every call moves all fields, so no
GPU is needed."""

import os
import re
import subprocess

from exploringsycl_amd import native

PKG = native.PKG_DIR

MAIN = r"""
#include <stdio.h>
#include <string.h>
#include "kernel_interface.h"
#include "kernel_interface_ext.h"
#include "tea_hip.h"

static double g_cells[1 << 16];
static int g_moves = 0;
extern "C" const char* tea_hip_last_error(void) { return ""; }
extern "C" int tea_hip_field(tea_hip_chunk*, int field, double** p, size_t*) {
  *p = g_cells + 32 * g_moves + field;
  return 0;
}
void die(int, const char*, const char*, ...) {}
%(stubs)s

static Chunk c;
static Settings s;
static ChunkExtension ext;
static void check(const char* call) {
  double* f[TEA_NUM_FIELDS];
  for (int k = 0; k < TEA_NUM_FIELDS; ++k) tea_hip_field(nullptr, k, &f[k], nullptr);
  if (c.p == f[TEA_FIELD_P] && c.u == f[TEA_FIELD_U] && c.r == f[TEA_FIELD_R] &&
      c.w == f[TEA_FIELD_W] && c.sd == f[TEA_FIELD_SD])
    return;
  printf("%%s\n", call);
}

int main() {
  c.ext = &ext;
  static int nb[4] = {-1, -1, -1, -1};
  c.neighbours = nb;
  for (int f = 0; f < 4; ++f) nb[f] = EXTERNAL_FACE;
  static bool exchange[NUM_FIELDS] = {};
  s.fields_to_exchange = exchange;
  s.num_states = 1;
  static State state[1] = {};
  double a = 0.0, b = 0.0, d = 0.0, e = 0.0, host[1];
  float norm[4] = {0.0f, 1.0f, 0.0f, 1.0f};
#define CALL(x) x; check(#x)
  CALL(run_set_chunk_data(&c, &s));
  CALL(run_set_chunk_state(&c, &s, state));
  CALL(run_store_energy(&c, &s));
  CALL(run_local_halos(&c, &s, 1));
  CALL(run_field_summary(&c, &s, &a, &b, &d, &e));
  CALL(run_cg_init(&c, &s, 1.0, 1.0, &a));
  CALL(run_cg_calc_w(&c, &s, &a));
  CALL(run_cg_calc_ur(&c, &s, 1.0, &a));
  CALL(run_cg_calc_p(&c, &s, 1.0));
  CALL(run_cheby_init(&c, &s));
  CALL(run_cheby_iterate(&c, &s, 1.0, 1.0));
  CALL(run_ppcg_init(&c, &s));
  CALL(run_ppcg_inner_iteration(&c, &s, 1.0, 1.0));
  CALL(run_jacobi_init(&c, &s, 1.0, 1.0));
  CALL(run_jacobi_iterate(&c, &s, &a));
  CALL(run_copy_u(&c, &s));
  CALL(run_calculate_residual(&c, &s));
  CALL(run_calculate_2norm(&c, &s, c.u, &a));
  CALL(run_finalise(&c, &s));
  CALL(run_mpcg_init(&c, &s, 1.0, 1.0, &a, &b));
  CALL(run_mpcg_calc_w(&c, &s, 1.0, 1, 1.0, 1, &a, &b));
  CALL(run_mpcg_calc_r(&c, &s, 1.0, &a, &b));
  CALL(run_mpcg_refresh(&c, &s, 1.0, 1, &a, &b, &d));
  CALL(run_fcg_attach(&c, &s, nullptr, 0, norm, 8, 1));
  CALL(run_fcg_attach_sweeps(&c, &s, 6, 8, 2));
  CALL(run_fcg_init(&c, &s, 1.0, 1.0, &a, &b));
  CALL(run_fcg_precondition(&c, &s, 0, &a));
  CALL(run_fcg_calc_w(&c, &s, 1.0, 1, 1.0, &a, &b));
  CALL(run_fcg_calc_r_precondition(&c, &s, 1.0, 0, &a, &b));
  CALL(run_read_u(&c, &s, host));
  return g_moves < 30;
}
"""


def test_every_call_republishes_the_addresses(tmp_path):
    header = re.sub(r"/\*.*?\*/", "", open(native.HEADER_PATH).read(), flags=re.S)
    stubs = []
    for name, args in re.findall(r"\bint (tea_hip_\w+)\(([^)]*)\)", header):
        if name != "tea_hip_field":
            stubs.append(f'extern "C" int {name}({args}) {{ return ++g_moves, 0; }}')
    stubs.append('extern "C" const char* tea_hip_kernel_name(int) { return ""; }')
    (tmp_path / "main.cpp").write_text(MAIN % {"stubs": "\n".join(stubs)})
    exe = str(tmp_path / "adapter")
    subprocess.run(
        ["g++", "-std=c++17", "-w", "-o", exe, str(tmp_path / "main.cpp"),
         os.path.join(PKG, "csrc", "kernel_interface_hip.cpp"), "-I", os.path.join(PKG, "host"),
         "-I", os.path.join(PKG, "csrc", "backend"), "-I", os.path.dirname(native.HEADER_PATH)],
        check=True)
    p = subprocess.run([exe], capture_output=True, text=True, timeout=30)
    assert p.returncode == 0
    assert p.stdout.split("\n") == [""], p.stdout
