"""The choices of kernel, tile and split (csrc/rules.hpp) on both sides of their lines, on the CPU: the header is
plain C++ and is compiled into a small program here."""
import pathlib
import shutil
import subprocess

import pytest

CSRC = pathlib.Path(__file__).resolve().parents[1] / "tsfm-zig_amd" / "csrc"

MAIN = r"""
#include <cstdio>
#include <cstring>
#include "rules.hpp"
using namespace tsfm::rules;
int main() {
    char what[32];
    while (scanf("%31s", what) == 1) {
        if (!strcmp(what, "attn")) {
            long rows; int n_q, n_k, mask, dense, rel, rope;
            if (scanf("%ld %d %d %d %d %d %d", &rows, &n_q, &n_k, &mask, &dense, &rel, &rope) != 7) return 1;
            AttnForm f = {rows, n_q, n_k, mask == 2 || mask == 3, mask == 5, mask == 4, mask == 1, dense != 0,
                          rel != 0, rope != 0};
            printf("%d\n", (int)attn_x3_pays(f, 256));
        } else if (!strcmp(what, "planes")) {
            long tokens, d_in, cols; int whole;
            if (scanf("%ld %ld %ld %d", &tokens, &d_in, &cols, &whole) != 4) return 1;
            printf("%d\n", (int)planes_pay(tokens, d_in, cols, whole != 0, 256));
        } else if (!strcmp(what, "split")) {
            long tokens, d_in, cols;
            if (scanf("%ld %ld %ld", &tokens, &d_in, &cols) != 3) return 1;
            const Split s = reduction_split((tokens + 63) / 64 * ((cols + 63) / 64), (int)(d_in / 16), d_in % 32 == 0,
                                            [] { return 256; });
            printf("%d %d\n", s.shares, s.steps);
        } else if (!strcmp(what, "splits")) {  // the most shares of 64 x 64 tiles any product has
            long most = 0;
            for (long blocks = 1; blocks < 2000; blocks++)
                for (int steps = 1; steps <= 512; steps++)
                    for (int pairs = 0; pairs < 2; pairs++) {
                        const Split s = reduction_split(blocks, steps, pairs != 0, [] { return 256; });
                        if (s.shares < 1 || s.steps * s.shares < steps || s.steps * (s.shares - 1) >= steps) return 2;
                        if (s.shares > 1 && s.shares * blocks > most) most = s.shares * blocks;
                    }
            printf("%ld\n", most);
        } else if (!strcmp(what, "keep")) {
            KeptWeights k;
            long tokens;
            while (scanf("%ld", &tokens) == 1) k.add(tokens);
            printf("%d\n", (int)k.pay());
        } else if (!strcmp(what, "big")) {
            long d_in, cus; int pre;
            if (scanf("%ld %d %ld", &d_in, &pre, &cus) != 3) return 1;
            printf("%d\n", (int)big_tiles_min(d_in, pre != 0, cus));
        }
    }
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("clang++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    d = tmp_path_factory.mktemp("rules")
    (d / "main.cpp").write_text(MAIN)
    subprocess.run([cxx, "-std=c++17", "-Wall", "-Werror", "-I", str(CSRC), str(d / "main.cpp"), "-o", str(d / "main")],
                   check=True)

    def ask(*words):
        out = subprocess.run([str(d / "main")], input=" ".join(str(w) for w in words), capture_output=True, text=True,
                             check=True).stdout
        return [int(x) for x in out.split()]

    return ask


FORMS = dict(plain=(0, 0, 0), dense=(1, 0, 0), t5=(0, 1, 0), rope=(0, 0, 1))
FULL, KEYS_ADDITIVE, CAUSAL, CAUSAL_KEYS, FULL_KEYS, DECODER = range(6)


@pytest.mark.parametrize("rows,n_q,mask,form,x3", [
    # one row per CU or fewer: only where the bf16x3 kernel measured faster, form by form
    (12, 64, KEYS_ADDITIVE, "rope", 0), (12, 66, KEYS_ADDITIVE, "rope", 1), (252, 109, FULL, "rope", 1),
    (12, 66, KEYS_ADDITIVE, "plain", 0), (12, 69, KEYS_ADDITIVE, "plain", 1), (252, 66, FULL, "t5", 0),
    (252, 128, KEYS_ADDITIVE, "t5", 1), (12, 129, KEYS_ADDITIVE, "t5", 0),
    (12, 80, KEYS_ADDITIVE, "dense", 0), (252, 144, KEYS_ADDITIVE, "dense", 0), (252, 128, FULL, "dense", 0),
    (252, 80, FULL_KEYS, "rope", 0), (12, 66, FULL_KEYS, "plain", 0), (12, 144, FULL_KEYS, "plain", 1),
    (252, 144, FULL_KEYS, "rope", 0), (12, 72, DECODER, "rope", 0), (12, 72, DECODER, "plain", 1),
    # more
    (264, 37, KEYS_ADDITIVE, "rope", 1), (264, 7, KEYS_ADDITIVE, "rope", 0), (264, 33, KEYS_ADDITIVE, "rope", 0),
    (768, 129, KEYS_ADDITIVE, "t5", 1), (264, 129, KEYS_ADDITIVE, "dense", 0), (516, 129, KEYS_ADDITIVE, "dense", 1),
    (504, 144, KEYS_ADDITIVE, "dense", 0), (264, 144, KEYS_ADDITIVE, "dense", 1),
    (768, 37, FULL_KEYS, "rope", 0), (264, 24, FULL_KEYS, "rope", 1), (504, 72, FULL_KEYS, "plain", 0),
    (384, 72, FULL_KEYS, "plain", 1), (264, 16, KEYS_ADDITIVE, "plain", 0), (516, 16, KEYS_ADDITIVE, "plain", 1),
    (384, 37, FULL, "plain", 0), (384, 37, KEYS_ADDITIVE, "plain", 1), (264, 32, DECODER, "rope", 1),
    # the causal masks
    (264, 109, CAUSAL, "rope", 0), (516, 95, CAUSAL_KEYS, "rope", 0), (516, 96, CAUSAL, "rope", 1)])
def test_short_row_attention_kernel(rules, rows, n_q, mask, form, x3):
    assert rules("attn", rows, n_q, 94 if mask == DECODER else n_q, mask, *FORMS[form]) == [x3]


@pytest.mark.parametrize("d_in,presplit,cus,tiles", [
    (768, 0, 256, 200), (512, 0, 256, 200), (768, 1, 256, 160), (512, 1, 256, 200), (1024, 1, 128, 80),
    (48, 0, 256, 256), (176, 0, 256, 256), (528, 0, 256, 200), (48, 0, 128, 128)])
def test_tiles_from_which_a_product_runs_on_the_big_ones(rules, d_in, presplit, cus, tiles):
    """The reductions that run on the f32 instruction (not of whole 32s) keep a full round of the small tiles, four a
    CU: 1100 to 1200 rows of the Chronos-2 patch embedding (48 values, 3072 columns) are 216 and 240 big tiles."""
    assert rules("big", d_in, presplit, cus) == [tiles]


@pytest.mark.parametrize("tokens,d_in,cols,whole,pre", [
    # long reductions that cannot be shared out: q/k/v products with RoPE
    (200, 4096, 1536, 1, 1), (768, 4096, 1536, 1, 1), (484, 3072, 2304, 1, 1), (545, 2048, 1536, 1, 1),
    (768, 1536, 1536, 1, 1), (545, 1536, 1536, 1, 0), (128, 2048, 6144, 1, 0), (64, 4096, 1536, 1, 0),
    (768, 768, 2304, 1, 0), (1928, 768, 2304, 1, 0), (1500, 1536, 1536, 1, 0),
    # the same without RoPE: shared out, or tiles enough
    (200, 4096, 1536, 0, 0), (545, 2048, 1536, 0, 0), (1205, 2048, 1536, 0, 1), (400, 2048, 6144, 0, 0),
    # by work and rows
    (1332, 1024, 3072, 1, 1), (1205, 1024, 3072, 0, 0), (999, 1024, 4096, 0, 0), (1332, 1024, 4096, 0, 1),
    (1500, 3072, 768, 0, 0), (2048, 768, 768, 0, 1), (2048, 512, 512, 0, 0), (2600, 1040, 2304, 0, 0)])
def test_presplit_operands(rules, tokens, d_in, cols, whole, pre):
    assert rules("planes", tokens, d_in, cols, whole) == [pre]


@pytest.mark.parametrize("tokens,d_in,cols,shares", [
    (33, 2048, 4096, 8), (8, 4096, 2048, 16), (17, 1024, 4096, 8),  # 512 workgroups, two a CU
    (545, 768, 768, 4), (528, 512, 1536, 2), (545, 768, 2304, 2),  # about 420
    (448, 256, 3 * 24 * 64, 1), (64, 256, 3 * 139 * 64, 2), (64, 256, 3 * 140 * 64, 1), (64, 240, 512, 1)])
def test_shares_of_a_reduction(rules, tokens, d_in, cols, shares):
    got, steps = rules("split", tokens, d_in, cols)
    assert got == shares and steps * got >= d_in // 16


def test_shares_cover_the_reduction_and_fit_the_fixed_array(rules):
    """Every share has steps to walk, and the partial sums of no product pass the 16 MiB array of
    tsfm_qkv_project_noalloc: at most 2 x 419 tiles of 64 x 64 floats, the figure in its header."""
    most = rules("splits")[0]
    assert most == 2 * 419 and most * 64 * 64 * 4 == 13729792 <= 16 << 20


@pytest.mark.parametrize("blocks,keep", [
    ([440, 94], 0), ([500] * 5, 0), ([1512, 564], 0), ([2016, 752], 0), ([1760, 376], 0), ([6512, 752], 0), ([2600], 0),
    ([767] * 8, 0), ([768, 768, 432], 0), ([768, 768, 768, 432], 1), ([1900, 940], 1), ([3024, 1128], 1), ([1024, 1024], 1)])
def test_split_weights_kept_for_a_forecast(rules, blocks, keep):
    """Only blocks of 768 tokens read the kept copy, so only they count for it."""
    assert rules("keep", *blocks) == [keep]
