"""What the kernel of gated and experts' products of few rows reads, walked on the CPU: its source, compiled for the host, over
operands that end where a page without access begins."""

import os
import re
import subprocess

import pytest

from mini_gpt_inference_amd.csrc import build

PROGRAM = r"""
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <sys/mman.h>
typedef uint16_t bf16_t;
typedef bf16_t ex_bf16x8_t __attribute__((ext_vector_type(8)));
typedef float ex_f32x4_t __attribute__((ext_vector_type(4)));
static struct { int x, y, z; } threadIdx, blockIdx;
struct Met {};                                // a thread's walk ends where the workgroup meets: behind it nothing is read from memory
#define __global__ static
#define __shared__ static
#define __launch_bounds__(threads)
#define address_space(number) aligned(1)
#define __syncthreads() throw Met()
#define __builtin_amdgcn_global_load_lds(from, to, bytes, offset, aux) memcpy((void*)(to), (const void*)(from), bytes)
#define __builtin_amdgcn_readfirstlane(v) (v)
#define __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, a, c, x, y, z) ((c) + (float)((w)[0] + (a)[0]))
#define EX_STEP STEP_OF_THE_SOURCE
#define EX_EPI_RELU2 1
template <bool FAST> float gated_value(float g, float u, int, float, float) { return g + u; }
static float relu_squared(float v) { return v; }
template <typename T> T from_float(float v) { return (T)v; }
KERNEL_OF_THE_SOURCE
static bf16_t* ends_at_a_page(size_t values) {
  const size_t page = 4096, bytes = values * 2, pages = (bytes + page - 1) / page * page;
  char* at = (char*)mmap(nullptr, pages + page, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
  if (at == MAP_FAILED || mprotect(at + pages, page, PROT_NONE)) exit(3);
  return (bf16_t*)(at + pages - bytes);
}
template <bool GATED, int STAGES, bool REST> void walk(int k, int rows, int o) {
  const bf16_t *a = ends_at_a_page((size_t)rows * k), *w = ends_at_a_page((size_t)(GATED ? 2 : 1) * o * k);
  float out[1];
  for (blockIdx.x = 0; blockIdx.x < (o + 15) / 16; ++blockIdx.x)
    for (threadIdx.x = 0; threadIdx.x < 256; ++threadIdx.x)
      try {
        grouped_few_rows_kernel<float, GATED, STAGES, REST>(a, k, nullptr, w, 0, nullptr, nullptr, out, o, nullptr, rows, o, k, 0, GATED ? 0 : -1, 0.f, 0.f);
      } catch (Met) {}
}
int main(int, char** argv) {
  const int k = atoi(argv[1]), rows = atoi(argv[2]), o = atoi(argv[3]);
  walk<true, 1, false>(k, rows, o), walk<true, 2, false>(k, rows, o), walk<false, 1, false>(k, rows, o), walk<false, 2, false>(k, rows, o);
  walk<true, 1, true>(k, rows, o), walk<false, 1, true>(k, rows, o), walk<false, 2, true>(k, rows, o);
}
"""


@pytest.fixture(scope="module")
def walk(tmp_path_factory):
    with open(os.path.join(build.HIP_DIR, "experts.hip"), encoding="utf-8") as fh:
        source = fh.read()
    kernel = re.search(r"template <typename OT, bool GATED, int STAGES, bool REST>\n__global__.*?\n}\n", source, re.S).group()
    step = re.search(r"#define EX_STEP (\d+)", source).group(1)
    text = PROGRAM.replace("STEP_OF_THE_SOURCE", step).replace("KERNEL_OF_THE_SOURCE", re.sub(r"asm volatile\([^;]*\);", ";", kernel))
    folder = tmp_path_factory.mktemp("walk")
    (folder / "walk.cpp").write_text(text)
    clang = build._find("clang++", ("/opt/rocm/llvm/bin",))
    subprocess.run([clang, "-O0", "-std=c++17", "-w", str(folder / "walk.cpp"), "-o", str(folder / "walk")], check=True)
    return str(folder / "walk")


@pytest.mark.parametrize("rows", [1, 5, 16])
@pytest.mark.parametrize("k", [8, 40, 56, 64, 72, 120, 320, 2120])
def test_reads_end_with_the_operands(walk, k, rows):
    """Inner sizes without a whole step of 64, of whole steps for some of the waves only, and with a rest."""
    assert subprocess.run([walk, str(k), str(rows), "33"]).returncode == 0
