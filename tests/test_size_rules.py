"""Rules on sizes that choose a route (csrc/size_rules.hpp), compiled by the host compiler.  No GPU."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "mamba_rs_amd", "csrc")


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    """rules("expression", args): the expression for every line of arguments a, b, c, d."""
    folder = tmp_path_factory.mktemp("rules")

    def run(expression, lines):
        exe, src = str(folder / "main"), str(folder / "main.cpp")
        with open(src, "w") as f:
            f.write(f'#include "size_rules.hpp"\n#include <cstdio>\nusing namespace mrs;\n'
                    f'int main() {{ long a, b, c, d; while (scanf("%ld %ld %ld %ld", &a, &b, &c, &d) == 4) printf("%ld\\n", (long)({expression})); }}\n')
        subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, "-o", exe, src], check=True)
        text = "".join(" ".join(map(str, line)) + "\n" for line in lines)
        return [int(v) for v in subprocess.run([exe], input=text, capture_output=True, text=True, check=True).stdout.split()]
    return run


def test_an_operand_that_is_not_there_lies_on_no_piece(rules):
    assert rules("in_pieces((const void *)a)", [(p, 0, 0, 0) for p in (0, 16, 4096, 8, 4098)]) == [0, 1, 1, 0, 0]


def test_slices_of_out_proj_are_those_of_the_rows_at_hand(rules):
    """A generation's buffers are made for 32 steps of all slots and used by shorter pieces: 13 slots of d_model 1024 and 11 or 12 steps are 48 tiles in four slices (in 32 steps, 112 in two), 64 of
    768 and four steps as well.  What a piece of any length takes is in the buffers, and slices never outgrow the chip or the sum behind them."""
    assert rules("mid_gemm_slices(a, (int)b, (int)c)", [(13 * 11, 1024, 2048, 0), (13 * 12, 1024, 2048, 0), (13 * 32, 1024, 2048, 0), (64 * 4, 768, 1536, 0), (64 * 32, 768, 1536, 0)]) == [4, 4, 2, 4, 1]
    lines = [(batch * T, dm, 2 * dm, batch * 32) for batch in (1, 3, 13, 64, 128) for dm in (64, 128, 320, 768, 1024, 1536, 2560, 4096) for T in range(2, 33)]
    slices, room = rules("mid_gemm_slices(a, (int)b, (int)c)", lines), rules("mid_gemm_parts_floats(d, (int)b, (int)c)", lines)
    for (rows, dm, _, _), n, r in zip(lines, slices, room):
        assert 1 <= n <= 4 and (n == 1 or n * rows * dm <= r) and r <= 512 * 64 * 64, (rows, dm, n, r)


def _columns(dm, ds=16):
    return (dm + 15) // 16 + 2 * ds


def test_conv_and_x_proj_are_one_launch_at_every_width_that_fits(rules):
    """Default hyperparameters, d_model 256 to 2560 in steps of 64: a prefill of many rows takes the one launch, one of some hundred rows of a model with enough
    channels has them in slices, and short ones keep two launches."""
    dims = range(256, 2561, 64)
    assert rules("conv_xproj_columns_ok(a)", [(_columns(dm), 0, 0, 0) for dm in dims]) == [1] * len(dims)
    assert rules("conv_xproj_columns_ok(a)", [(xd, 0, 0, 0) for xd in (32, 33, 34, 194, 196, 208)]) == [0] * 6
    assert rules("conv_xproj_columns_ok(a)", [(xd, 0, 0, 0) for xd in (36, 48, 52, 188, 192)]) == [1] * 5
    form = "conv_xproj_form(a, b, c, d)"
    for B, T in ((8, 2048), (4, 4096), (1, 7000), (300, 5)):
        assert rules(form, [(B, T, 2 * dm, _columns(dm)) for dm in dims]) == [1] * len(dims)
    assert all((f >= 2) == (dm >= 512) and f for dm, f in zip(dims, rules(form, [(2, 1664, 2 * dm, _columns(dm)) for dm in dims])))
    assert rules(form, [(1, 300, 2 * dm, _columns(dm)) for dm in dims]) == [0] * len(dims)


def test_slices_of_the_channels_fit_their_room_and_the_chip(rules):
    """The shares of x_proj's products in f32 take at most the bytes of u in 16 bits, a slice has at least two pieces of channels but perhaps the last, and all workgroups
    run at once."""
    lines = [(1, 32 * tiles - 7, 2 * dm, _columns(dm, ds)) for ds in (8, 16, 32, 64) for dm in range(128, 2561, 32) for tiles in range(1, 131)
             if _columns(dm, ds) % 4 == 0 and 33 <= _columns(dm, ds) <= 192]
    forms = rules("conv_xproj_form(a, b, c, d)", lines)
    sliced = 0
    for (_, T, di, xd), f in zip(lines, forms):
        if f >= 2:
            sliced += 1
            assert f <= 16 and f * xd * 4 <= di * 2 and f * ((T + 31) // 32) <= 256 and di // 64 >= 2 * f, (T, di, xd, f)
    assert sliced > 1000


def test_out_proj_is_asked_for_ahead_only_where_it_stays_in_the_l2(rules):
    """Eight dies have 4 MB of L2 each: few rows ask ahead for what fits, many also where it is a little more, and nobody for much more."""
    ahead = [(2 * dm * 2 * dm, rows) for rows in (3, 4, 8, 16, 64) for dm in (1536, 2048, 2560, 2816, 3072, 3328, 3584)]
    want = [nbytes <= (28 if rows < 8 else 40) * 2 ** 20 for nbytes, rows in ahead]
    assert rules("asks_out_proj_ahead(a, (int)b)", [(nbytes, rows, 0, 0) for nbytes, rows in ahead]) == want
    assert not any(w for w, (nbytes, _) in zip(want, ahead) if nbytes > 40 * 2 ** 20) and all(w for w, (nbytes, _) in zip(want, ahead) if nbytes <= 25 * 2 ** 20)


def test_layers_whose_weights_come_through_the_last_cache(rules):
    """All of them while they fit beside the states (240 MB), else no more than leave the states their room, and never fewer than none."""
    mb = 2 ** 20
    cases = [(24, 7 * mb, 3 * mb), (24, 7 * mb, 72 * mb), (24, 7 * mb, 73 * mb), (24, 13 * mb, 3 * mb), (24, 13 * mb, 50 * mb), (24, 7 * mb, 400 * mb), (8, 78 * mb, 40 * mb), (64, 0, 300 * mb)]
    assert rules("layers_in_cache((int)a, b, c)", [(*c, 0) for c in cases]) == [24, 24, 21, 16, 13, 0, 2, 0]
    assert rules("streams_in_proj(a, (int)b)", [(240 * mb, 4, 0, 0), (240 * mb + 1, 4, 0, 0), (10 ** 9, 48, 0, 0), (10 ** 9, 49, 0, 0)]) == [0, 1, 1, 0]


def test_the_own_chain_takes_every_row_count_up_to_d_model_1536(rules):
    assert rules("own_chain_to_the_last_row(a, b)", [(dm, 2 * dm, 0, 0) for dm in (64, 768, 1024, 1536, 1792, 2560)] + [(2048, 2048, 0, 0)]) == [1, 1, 1, 1, 0, 0, 1]


def test_the_mamba3_step_has_whole_waves(rules):
    """Every head that an engine takes: headdim x d_state / 4 threads, a multiple of 64 of at most 1024."""
    heads = [(hd, ds) for ds in (4, 8, 16, 32, 64, 128, 256) for hd in range(4, 257) if hd * (ds // 4) % 64 == 0 and hd * (ds // 4) <= 1024]
    for batch, nh in ((1, 24), (8, 24), (191, 1), (3, 64)):
        rows = rules("m3_step_rows(a / 1000, a % 1000, b, c, d)", [(1000 * batch + nh, hd, ds, ds // 2) for hd, ds in heads])
        for (hd, ds), r in zip(heads, rows):
            assert r == (4 if batch * nh >= 192 and ds == 64 and hd % 16 == 0 else 1) and hd * (ds // 4) // r % 64 == 0 and hd * (ds // 4) // r >= min(ds, 64), (batch, nh, hd, ds, r)


def test_f32_prefills_of_many_rows_read_their_weights_as_they_came(rules):
    """Engines of five rows and more have transposed copies for their decode; the library is handed them in a prefill only where that is ahead at nearly every size."""
    assert rules("f32_prefill_transposed(a, 2 * a, b)", [(dm, rbr, 0, 0) for rbr in (0, 1) for dm in (192, 768, 1024, 2048, 2560)]) == [0, 0, 0, 0, 1, 1, 1, 1, 1, 1]


def test_rows_of_the_f32_chain(rules):
    dims = (192, 256, 768, 1024, 1536, 2560)
    assert rules("own_f32_chain_rows(a, b, false)", [(dm, 2 * dm, 0, 0) for dm in dims]) == [128, 128, 128, 64, 48, 48]
    assert rules("own_f32_chain_rows(a, b, true)", [(dm, 2 * dm, 0, 0) for dm in dims]) == [96, 96, 48, 48, 48, 48]
