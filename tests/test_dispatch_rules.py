"""The rules that choose a kernel from a call's sizes (csrc/qd_dispatch.h), compiled for
the host: at sizes measured on both sides, on 256 compute units, the faster one."""
import ctypes
import os
import subprocess

import pytest

from conftest import ROOT

CUS = 256
SHIM = r"""
#include "qd_dispatch.h"
extern "C" {
int shares_fused(int heads, int seqlen, int tokens, int cus) { return qd::prefill_shares_fused(heads, seqlen, tokens, cus); }
int shares_split(int heads, int seqlen, int tokens, int cus) { return qd::prefill_shares_split(heads, seqlen, tokens, cus); }
int merges_by_wave(int heads, int tokens, int splits) { return qd::prefill_merges_by_wave(heads, tokens, splits); }
int exact_two_rows(int tokens, int n, int k, int cus) { return qd::exact_two_rows(tokens, n, k, cus); }
int short_tile(long long rows, int tokens, int k, int paired, int res, int scalar, int cus) {
  return (int)qd::short_tile(rows, tokens, k, paired, res, scalar, cus);
}
int ring_two_slices(long long tiles, int cus) { return qd::ring_two_slices(tiles, cus); }
long long ring_two_slice_bytes(int outputs, int cus) { return (long long)qd::ring_two_slice_bytes(outputs, cus); }
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("rules")
    src, lib = tmp / "shim.cpp", tmp / "shim.so"
    src.write_text(SHIM)
    csrc = os.path.join(ROOT, "llm-inference-diy_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-I", csrc, "-o", str(lib), str(src)],
                   check=True)
    return ctypes.CDLL(str(lib))


@pytest.mark.parametrize("heads,pos0,tokens,scan_us,shared_us", [
    (1, 0, 56, 3.89, 7.35), (1, 0, 224, 4.91, 12.85), (2, 164, 60, 4.80, 12.89), (4, 0, 56, 4.07, 7.61),
    (4, 0, 128, 5.97, 9.17), (4, 0, 224, 10.44, 12.87), (4, 124, 100, 7.09, 12.90), (8, 0, 56, 5.63, 7.65),
    (8, 0, 96, 7.51, 9.08), (8, 0, 128, 9.34, 9.21), (8, 68, 60, 6.14, 9.22), (12, 0, 64, 7.39, 7.80),
    (12, 0, 96, 10.67, 9.11), (12, 164, 60, 9.80, 12.96), (12, 124, 100, 13.91, 12.95), (16, 0, 48, 7.31, 7.56),
    (16, 0, 56, 8.81, 7.72), (16, 0, 128, 16.34, 9.31), (20, 0, 56, 10.24, 7.78), (20, 194, 30, 9.85, 12.97),
    (24, 0, 40, 8.79, 7.51), (32, 0, 20, 7.03, 7.11), (32, 0, 32, 8.78, 7.34), (32, 64, 16, 6.09, 8.88),
    (64, 0, 24, 11.77, 7.36), (64, 64, 8, 6.02, 8.85), (64, 0, 128, 56.27, 16.18)])
def test_fused_prompt_attention_takes_the_faster_form(rules, heads, pos0, tokens, scan_us, shared_us):
    assert bool(rules.shares_fused(heads, pos0 + 1, tokens, CUS)) == (shared_us < scan_us)


@pytest.mark.parametrize("heads,pos0,tokens,scan_us,shared_us", [
    (1, 1000, 48, 11.9, 13.7), (1, 4000, 48, 35.9, 27.9), (4, 300, 64, 14.78, 15.76), (4, 1000, 12, 10.73, 11.98),
    (4, 1000, 24, 15.50, 12.44), (4, 4000, 8, 12.86, 10.03), (8, 1000, 6, 8.1, 9.1), (8, 1000, 12, 10.6, 10.5),
    (8, 2000, 6, 8.87, 9.37), (12, 600, 32, 19.3, 13.5), (16, 128, 64, 24.86, 20.46), (16, 300, 8, 8.51, 10.20),
    (16, 1000, 4, 7.69, 9.24), (16, 1000, 6, 8.76, 9.24), (16, 1000, 8, 9.83, 9.32), (16, 2000, 6, 14.54, 13.38),
    (16, 8000, 6, 54.63, 39.65), (20, 1000, 6, 11.50, 12.66), (20, 1000, 12, 17.1, 16.1), (24, 1000, 6, 12.26, 13.44),
    (32, 600, 6, 10.43, 12.53), (32, 1000, 12, 22.7, 16.7), (64, 300, 6, 11.06, 14.76), (64, 300, 8, 12.27, 14.82),
    (64, 1000, 8, 35.7, 19.6), (128, 128, 16, 20.15, 24.10), (128, 1000, 8, 76.6, 30.4)])
def test_split_prompt_attention_takes_the_faster_form(rules, heads, pos0, tokens, scan_us, shared_us):
    assert bool(rules.shares_split(heads, pos0 + 1, tokens, CUS)) == (shared_us < scan_us)


def test_up_to_five_queries_of_split_plans_are_scanned(rules):
    for heads in (1, 4, 16, 256, 4096):
        for tokens in (1, 2, 5):
            assert not rules.shares_split(heads, 100000, tokens, CUS)


@pytest.mark.parametrize("heads,tokens,splits,group_us,wave_us", [
    (1, 1, 63, 6.14, 7.44), (4, 1, 64, 6.30, 8.73), (4, 64, 64, 20.31, 23.84), (4, 256, 64, 48.50, 52.32),
    (8, 1, 32, 6.00, 7.23), (8, 128, 32, 31.06, 34.97), (12, 6, 21, 10.3, 11.3), (16, 1, 16, 6.16, 6.52),
    (16, 16, 16, 11.31, 12.25), (16, 64, 16, 32.82, 34.76), (16, 128, 16, 52.02, 53.56), (16, 256, 16, 89.70, 88.43),
    (20, 256, 12, 91.1, 86.6), (32, 256, 8, 80.7, 74.5), (64, 32, 4, 31.6, 29.7), (128, 48, 2, 82.7, 73.2)])
def test_prompt_merge_takes_the_faster_form(rules, heads, tokens, splits, group_us, wave_us):
    assert bool(rules.merges_by_wave(heads, tokens, splits)) == (wave_us < group_us)


@pytest.mark.parametrize("tokens,n,k,two_rows_us,matrix_us", [
    (1, 16, 8192, 6.55, 13.40), (4, 16, 8192, 11.34, 13.33), (1, 1024, 7176, 8.15, 13.03), (4, 2048, 7176, 13.36, 14.14),
    (1, 2048, 8192, 11.32, 15.79), (2, 2048, 7680, 10.49, 14.86), (1, 4096, 8192, 20.42, 17.64),
    (4, 4096, 7176, 24.55, 15.59), (5, 4096, 8192, 36.91, 16.91), (5, 2048, 7176, 16.19, 14.21), (4, 6144, 2048, 9.1, 10.3),
    (4, 2048, 5504, 10.6, 11.3), (6, 2048, 5504, 12.7, 11.2), (16, 2048, 2048, 10.4, 6.2),
    (5, 98, 1928, 5.43, 6.02), (5, 6, 5400, 9.15, 10.15), (6, 3, 1416, 4.07, 4.79), (6, 90, 1352, 4.50, 4.76),
    (5, 15, 304, 2.91, 2.98), (5, 176, 3176, 8.85, 7.00), (6, 10219, 936, 8.90, 10.04), (5, 11934, 416, 6.32, 8.08), (6, 6931, 624, 6.77, 6.04),
    (6, 11228, 128, 5.74, 5.20), (5, 8488, 1296, 10.64, 10.33), (6, 9997, 240, 5.63, 6.76), (6, 12892, 1088, 12.31, 11.34),
    (8, 11530, 440, 7.03, 7.97), (7, 23427, 504, 11.01, 12.48), (8, 11773, 552, 8.57, 7.96), (7, 11682, 8, 5.42, 4.31)])
def test_exact_product_takes_the_faster_kernel(rules, tokens, n, k, two_rows_us, matrix_us):
    assert bool(rules.exact_two_rows(tokens, n, k, CUS)) == (two_rows_us < matrix_us)


@pytest.mark.parametrize("tokens,n,k,paired,res,us", [   # 64 x 64, 32 x 16, 32 x 32, 32 x 64, 64 x 128
    (1, 40000, 64, 0, 0, (7.86, 12.43, 12.60, 12.95, 10.23)), (32, 20000, 128, 0, 0, (7.01, 12.74, 8.88, 8.86, 8.05)),
    (1, 20000, 512, 0, 0, (9.12, 10.14, 10.34, 10.64, 10.90)), (16, 40000, 512, 0, 0, (15.28, 18.60, 18.75, 20.22, 18.07)),
    (1, 10000, 512, 1, 0, (9.06, 10.83, 10.98, None, 11.52)), (16, 15000, 512, 1, 0, (11.00, 15.74, 15.84, None, 12.98)),
    (1, 64, 2048, 0, 0, (9.33, 4.80, 5.29, 6.84, 11.35)), (16, 2048, 5504, 0, 0, (20.09, 9.47, 10.32, 13.17, 25.00)),
    (100, 2048, 2048, 0, 0, (10.14, 9.47, 6.63, 7.73, 12.64)), (100, 6144, 2048, 0, 0, (10.99, 23.15, 15.26, 13.48, 12.86)),
    (64, 6144, 2048, 0, 0, (10.34, 13.72, 11.79, 8.31, 12.64)), (32, 6144, 2048, 0, 0, (10.19, 10.21, 7.74, 7.79, 12.21)),
    (100, 5504, 2048, 1, 0, (23.69, 47.51, 34.52, None, 18.38)), (100, 2048, 5504, 0, 0, (20.47, 15.86, 11.23, 14.04, 26.90)),
    (127, 11008, 2048, 0, 0, (23.94, 56.21, 37.28, 28.45, 19.38)), (65, 40000, 2048, 0, 0, (68.11, 109.84, 78.89, 70.53, 47.15)),
    (200, 1000, 2048, 1, 0, (10.72, 17.28, 11.38, None, 13.46)), (160, 2048, 1024, 0, 0, (7.05, 10.48, 8.59, 6.05, 8.98)),
    (48, 1536, 512, 0, 0, (5.18, 4.11, 4.27, 4.60, 6.27)), (400, 1000, 1024, 0, 0, (7.13, 12.50, 8.14, 5.96, 8.88)),
    (48, 6144, 64, 0, 1, (5.37, 7.71, 5.97, 4.32, 5.64)), (16, 20000, 512, 0, 1, (11.79, 10.48, 10.74, 10.98, 11.50)),
    (32, 20000, 512, 0, 1, (14.91, 15.19, 11.08, 11.29, 12.34)), (127, 20000, 256, 0, 1, (20.34, 47.43, 26.96, 16.10, 13.15)),
    (100, 2048, 5504, 0, 1, (22.97, 16.26, 11.54, 14.38, 28.60)), (256, 2048, 2048, 0, 1, (11.61, 17.70, 11.39, 8.07, 14.24))])
def test_short_product_takes_the_fastest_tile(rules, tokens, n, k, paired, res, us):
    took = us[rules.short_tile(ctypes.c_longlong(n * (1 + paired)), tokens, k, paired, res, 0, CUS)]
    assert took is not None and took <= 1.05 * min(t for t in us if t is not None)


@pytest.mark.parametrize("tokens,n,k,paired,res,us", [   # the same tiles, y rows an odd number of elements apart
    (1367, 2010, 64, 0, 0, (10.15, 46.75, 27.64, 19.76, 13.78)), (559, 7218, 128, 0, 0, (14.08, 68.30, 40.18, 25.78, 18.01)),
    (231, 9978, 192, 0, 0, (11.61, 43.32, 28.64, 18.56, 14.61)), (403, 5123, 448, 0, 0, (14.77, 43.55, 27.18, 19.84, 17.18)),
    (1375, 1722, 512, 0, 0, (14.96, 48.18, 30.32, 20.38, 17.17)), (34, 9182, 128, 0, 1, (6.39, 13.00, 10.50, 9.00, 8.85)),
    (426, 5067, 64, 0, 1, (15.58, 45.41, 26.65, 20.14, 20.43)), (1301, 1901, 128, 0, 1, (16.89, 52.81, 29.97, 20.24, 20.25))])
def test_short_product_with_unaligned_outputs_takes_the_fastest_tile(rules, tokens, n, k, paired, res, us):
    took = us[rules.short_tile(ctypes.c_longlong(n * (1 + paired)), tokens, k, paired, res, 1, CUS)]
    assert took <= 1.05 * min(us)


@pytest.mark.parametrize("n,tokens,one_us,two_us", [   # us a layer of the whole prompt, both products so
    (2048, 1022, 237.6, 221.7), (4096, 510, 337.0, 304.5), (1024, 2046, 264.3, 247.9), (2048, 1100, 258.7, 275.4),
    (2048, 1300, 285.5, 306.1), (2048, 1920, 303.3, 330.3)])
def test_two_slices_of_k_where_both_run_at_once(rules, n, tokens, one_us, two_us):
    tiles = -(-n // 128) * -(-tokens // 128)
    assert bool(rules.ring_two_slices(ctypes.c_longlong(tiles), CUS)) == (two_us < one_us)


@pytest.mark.parametrize("cus", [256, 255, 304, 64])
def test_two_slices_of_k_fit_their_workspace(rules, cus):
    rules.ring_two_slice_bytes.restype = ctypes.c_longlong
    have = rules.ring_two_slice_bytes(128 * 128, cus)
    for wide in range(1, cus + 1):
        for high in range(1, cus // wide + 1):
            if rules.ring_two_slices(ctypes.c_longlong(wide * high), cus):
                assert 2 * (128 * wide) * (128 * high) * 4 <= have
