"""CPU tests of the C-ABI boundary: the built library loads and exports every
function that include/*.h declares (no compute call without a GPU)."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_functions():
    names = set()
    for fn in os.listdir(os.path.join(ROOT, "include")):
        if not fn.endswith(".h"):
            continue
        text = open(os.path.join(ROOT, "include", fn)).read()
        text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
        for m in re.finditer(r"\b(tc_[a-z0-9_]+)\s*\(", text):
            names.add(m.group(1))
    return sorted(names)


def test_header_declares_entry_points():
    names = declared_functions()
    for must in ("tc_gemv", "tc_gemm", "tc_gemv_dual", "tc_moe_ffn", "tc_quantize_act", "tc_block_isums"):
        assert must in names


def test_library_exports_every_declared_symbol():
    import tc_hip
    lib = tc_hip.load_library()
    missing = [n for n in declared_functions() if not hasattr(lib, n)]
    assert not missing, missing
    assert set(declared_functions()) == set(tc_hip.SIGNATURES)


def test_no_device_is_reported_cleanly():
    import tc_hip
    import torch
    if torch.cuda.is_available():
        pytest.skip("a GPU is present")
    lib = tc_hip.load_library()
    assert lib.tc_available() == 0
    rc = lib.tc_gemv(12, None, None, None, 1, 1, 256, None)
    assert rc == tc_hip.TC_E_UNSUPPORTED
    assert b"gfx950" in lib.tc_last_error()


def test_row_bytes():
    import tc_hip
    lib = tc_hip.load_library()
    assert lib.tc_row_bytes(12, 3584) == 14 * 144
    assert lib.tc_row_bytes(8, 4096) == 128 * 34
    assert lib.tc_row_bytes(14, 18944) == 74 * 210
    assert lib.tc_row_bytes(18, 3584) == 14 * 98
    assert lib.tc_row_bytes(11, 256) == 110
    assert lib.tc_row_bytes(10, 256) == 84
    assert lib.tc_row_bytes(9, 256) == 0  # Q8_1: not a weight type here


def test_type_ids_and_block_geometry():
    """The header's TC_* type ids are the binding's, and each type's row size
    is its GGUF block geometry as the GGUF reader's own table gives it (that
    table is checked against the reference loader in test_gguf.py). IQ2_XXS
    (16) and the reference's own formats are not weight types here."""
    import tc_hip
    lib = tc_hip.load_library()
    text = open(os.path.join(ROOT, "include", "tc_qmatmul.h")).read()
    enum = dict((m.group(1), int(m.group(2))) for m in re.finditer(r"\bTC_([A-Z0-9_]+) = (\d+)", text)
                if not m.group(1).startswith("E_") and m.group(1) != "OK")
    assert {k: v for k, v in enum.items() if k in tc_hip.TYPES} == tc_hip.TYPES
    assert set(tc_hip.TYPES) <= set(enum)
    for name, t in tc_hip.TYPES.items():
        bs, ts = lib.tc_gguf_block_size(t), lib.tc_gguf_type_size(t)
        assert (bs, ts) == (tc_hip.BLOCK_SIZE[t], tc_hip.TYPE_SIZE[t]), name
        assert lib.tc_row_bytes(t, 18944) == 18944 // bs * ts, name
        assert lib.tc_row_bytes(t, 3584) == 3584 // bs * ts, name
    for t in (0, 1, 16, 142, 143, 200):
        assert lib.tc_row_bytes(t, 256) == 0, t


def test_reference_interface_header_compiles_and_links(tmp_path):
    """include/tc_int8gemm.hpp (the reference's tinycoder::gpu interface over
    the C ABI) compiles as C++17, links against the library, and reports no
    device and refuses calls cleanly on a machine without a GPU."""
    import shutil
    import subprocess
    import tc_hip
    import torch
    if torch.cuda.is_available():
        pytest.skip("a GPU is present")
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no host C++ compiler")
    lib = tc_hip.load_library()
    so = lib._name
    src = tmp_path / "iface.cpp"
    src.write_text(
        '#include "tc_int8gemm.hpp"\n'
        "int main() {\n"
        "  namespace g = tinycoder::gpu;\n"
        "  if (g::int8GemmAvailable()) return 2;\n"
        "  if (g::int8Gemv(12, nullptr, nullptr, nullptr, 1, 1, 256, nullptr)) return 3;\n"
        "  if (g::int8Gemm(12, nullptr, nullptr, nullptr, 16, 1, 256, 1, nullptr)) return 4;\n"
        "  if (g::int8GemvDualIQ2XS(nullptr, nullptr, nullptr, nullptr, nullptr, 1, 256, nullptr)) return 5;\n"
        "  return 0;\n"
        "}\n")
    exe = tmp_path / "iface"
    subprocess.run([gxx, "-std=c++17", "-I", os.path.join(ROOT, "include"), str(src), so,
                    "-Wl,-rpath," + os.path.dirname(so), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stderr)


def test_cpp_interface_driver_without_gpu():
    """The C++ interface driver (tests/cpp, built from include/tc_int8gemm.hpp
    and include/tc_simd_matmul.hpp against the library) loads, and without a
    GPU every call reports false and writes nothing."""
    import numpy as np
    import torch
    if torch.cuda.is_available():
        pytest.skip("a GPU is present")
    import iface
    d = iface.load()
    assert d.drv_int8GemmAvailable() == 0
    assert d.drv_int8Gemv(12, None, None, None, 1, 1, 256, None) == 0
    assert d.drv_int8Gemm(12, None, None, None, 16, 1, 256, 1, None) == 0
    w = np.zeros(144, np.uint8)
    x = np.zeros(256, np.float32)
    out = np.full(1, 7.0, np.float32)
    for t in (12, 11, 14, 13, 23, 20, 8):
        assert d.drv_matMulVecBatch_SIMD(t, w.ctypes.data, x.ctypes.data, 1, 1, 256, out.ctypes.data, None) == 0
    assert out[0] == 7.0


def _compile_and_run(tmp_path, source, *args):
    """A host program over the library's internal headers and functions."""
    import shutil
    import subprocess
    import tc_hip
    import torch  # noqa: F401  (its HIP runtime's folder, for the library)
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no host C++ compiler")
    src = tmp_path / "prog.cpp"
    src.write_text(source)
    exe = tmp_path / "prog"
    so = tc_hip.load_library()._name
    subprocess.run([gxx, "-std=c++17", "-I", os.path.join(ROOT, "tinycoder-inference_amd", "csrc"), str(src), *args,
                    so, "-Wl,-rpath," + os.path.dirname(so), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)


def test_reserved_scratch_covers_every_route(tmp_path):
    """tc_gemv_reserve's sizes cover what any tc_gemv or tc_gemm call of at most
    the reserved tokens and columns asks of the two buffers, over all types,
    token counts around every tile width, narrow to wide inputs and rows up
    to the documented bound (such a call must not replace a buffer whose address
    a graph holds)."""
    import tc_hip
    types = ", ".join(str(t) for t in tc_hip.TYPES.values())
    _compile_and_run(tmp_path, r"""
#include <stdint.h>
#include <stdio.h>
namespace tc {
size_t mfma_scratch(int, uint32_t, uint32_t, uint32_t, int, size_t *);
size_t reserve_scratch(uint32_t, uint32_t, int, size_t *);
uint32_t gemv_max_tokens(int, uint32_t);
}
int main() {
    const uint32_t tokens[] = {1, 2, 3, 4, 5, 6, 7, 8, 9, 32, 33, 64, 65, 100, 128, 129, 256, 257, 333, 1000, 2048, 6000};
    const uint32_t cols[] = {256, 2304, 4096, 8192, 14336, 18944, 28672};
    const uint32_t rows[] = {1, 255, 256, 3584, 18944, 19712, 128256, 152064, 1u << 20};
    const int types[] = {""" + types + r"""};
    for (uint32_t rs : tokens)
        for (uint32_t rc : cols) {
            size_t ract = 0;
            const size_t raux = tc::reserve_scratch(rs, rc, 256, &ract);
            for (uint32_t s : tokens)
                for (uint32_t c : cols)
                    for (uint32_t n : rows)
                        for (int t : types) {
                            if (s > rs || c > rc || tc::gemv_max_tokens(t, c) == 0) continue;
                            size_t act = 0;
                            const size_t aux = tc::mfma_scratch(t, s, n, c, 256, &act);
                            if (act <= ract && aux <= raux) continue;
                            printf("reserved %u x %u: %zu, %zu; type %d, %u tokens, %u x %u: %zu, %zu\n", rs, rc, ract,
                                   raux, t, s, n, c, act, aux);
                            return 1;
                        }
        }
    return 0;
}
""")


def test_scratch_growth_rule(tmp_path):
    """Buffers that a graph may use are kept when they grow, and the kept ones
    stay smaller than the one in use; a failed growth leaves a buffer as it was
    unless the call cannot do without it."""
    _compile_and_run(tmp_path, r"""
#include <set>
#include "tc_scratch.hpp"
struct Mem {
    size_t *room;
    std::set<void *> *live, *gone;
    void *alloc(size_t n) {
        if (n > *room) return nullptr;
        void *p = new char;
        live->insert(p);
        return p;
    }
    void release(void *p) {
        live->erase(p);
        gone->insert(p);
        *room = 1000;
    }
};
#define CHECK(c) do { if (!(c)) return __LINE__ % 256; } while (0)
int main() {
    size_t room = 1 << 30;
    std::set<void *> live, gone;
    Mem m{&room, &live, &gone};
    tc::Scratch s;
    CHECK(tc::scratch_grow(s, 100, false, true, m) && s.bytes == 100 && !s.held);
    void *p = s.p;
    CHECK(tc::scratch_grow(s, 200, false, true, m) && s.bytes == 200 && gone.count(p));  // no graph: given back
    p = s.p;
    CHECK(tc::scratch_grow(s, 150, true, true, m) && s.p == p && s.held);  // recorded
    CHECK(tc::scratch_grow(s, 210, false, true, m) && s.p != p && s.bytes == 400 && live.count(p) && !s.held);
    p = s.p;
    CHECK(tc::scratch_grow(s, 500, true, true, m) && live.count(p) && s.held);  // grown while recording
    p = s.p;
    room = 0;
    CHECK(!tc::scratch_grow(s, 5000, false, true, m) && s.p == p && s.held);  // held: kept at any rate
    room = 1200;
    CHECK(tc::scratch_grow(s, 1100, false, true, m) && s.bytes == 1100 && live.count(p));  // twice does not fit
    p = s.p;
    room = 0;
    CHECK(!tc::scratch_grow(s, 1500, false, false, m) && s.p == p && s.bytes == 1100);  // optional: left alone
    CHECK(tc::scratch_grow(s, 900, false, false, m) && s.p == p);
    CHECK(!tc::scratch_grow(s, 1500, false, true, m) && gone.count(p) && s.p == nullptr && s.bytes == 0);
    CHECK(tc::scratch_grow(s, 1000, false, true, m) && s.bytes == 1000);
    return 0;
}
""")


def test_route_by_measured_times(tmp_path):
    """Calls of few tokens that the decode kernel was measured to serve faster
    keep it, and the gains of the matrix-core route stay (times in us, decode
    kernel against matrix cores)."""
    import tc_hip
    few = [("Q5_0", 4, 18944, 2048, 18, 30), ("Q5_0", 5, 18944, 2048, 20, 30), ("Q5_0", 4, 8192, 4096, 19, 28),
           ("Q5_0", 6, 32768, 1536, 23, 30), ("Q5_0", 2, 2560, 14336, 23, 34), ("IQ4_NL", 2, 3584, 13824, 21, 30),
           ("IQ4_NL", 4, 8192, 4096, 22, 27), ("IQ2_XS", 5, 32768, 3072, 37, 45), ("Q6_K", 2, 2560, 14336, 20, 27),
           ("Q6_K", 4, 2560, 8192, 21, 24), ("Q5_K", 6, 5120, 8192, 19, 24), ("Q5_K", 8, 3584, 10240, 24, 25),
           ("Q4_K", 4, 2560, 18944, 18, 23), ("IQ4_XS", 5, 3584, 13824, 21, 26), ("IQ4_XS", 6, 5120, 10240, 26, 28),
           ("Q6_K", 8, 3584, 18944, 137, 33), ("Q4_K", 8, 3584, 18944, 45, 26), ("IQ4_NL", 8, 3584, 18944, 163, 41),
           ("IQ4_NL", 5, 18944, 3584, 108, 38), ("Q6_K", 3, 256, 18944, 33, 21), ("Q5_K", 7, 5120, 11008, 36, 24)]
    prompt = [("IQ4_XS", 9, 8192, 2048, 15, 19), ("IQ4_XS", 9, 8192, 4096, 21, 27), ("IQ4_XS", 11, 4096, 1280, 14, 16),
              ("Q2_K", 9, 4096, 4096, 16, 17), ("IQ2_XS", 9, 8192, 2048, 22, 27), ("IQ4_XS", 9, 8192, 512, 13, 11),
              ("IQ4_XS", 14, 4096, 2560, 20, 16), ("IQ4_XS", 9, 12288, 3072, 27, 23), ("Q2_K", 9, 256, 256, 14, 8),
              ("Q2_K", 10, 4096, 4096, 18, 17), ("IQ2_XS", 9, 7168, 2304, 45, 24), ("Q5_0", 9, 18944, 3584, 150, 40)]
    rows = [f"{{{int(f is few)}, {tc_hip.TYPES[t]}, {s}, {n}, {k}, {int(mf < dec)}}}"
            for f in (few, prompt) for t, s, n, k, dec, mf in f]
    _compile_and_run(tmp_path, r"""
#include <stdint.h>
#include <stdio.h>
namespace tc {
bool few_tokens_mfma(int, uint32_t, uint32_t, uint32_t, int);
bool prompt_mfma(int, uint32_t, uint32_t, uint32_t);
}
int main() {
    const uint32_t c[][6] = {""" + ", ".join(rows) + r"""};
    for (auto &r : c) {
        const bool m = r[0] ? tc::few_tokens_mfma(int(r[1]), r[2], r[3], r[4], 256)
                            : tc::prompt_mfma(int(r[1]), r[2], r[3], r[4]);
        if (m == bool(r[5])) continue;
        printf("type %u, %u tokens, %u x %u: matrix cores %d\n", r[1], r[2], r[3], r[4], int(m));
        return 1;
    }
    return 0;
}
""")
