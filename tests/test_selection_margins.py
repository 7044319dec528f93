"""The margins by which a whole-vocabulary row's selection decides (head_kernel's tables of weights
in fixed point, head_pick_kernel's comparisons), from the constants of the source: no GPU."""
import os
import re

import numpy as np

SOURCE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tabby_amd", "csrc",
                      "tabby_sampler.hip")


def _constants():
    text = open(SOURCE).read()
    env = {}
    for name in ("kTableBins", "kWeightBits", "kTableError", "kPickAdds"):
        m = re.search(rf"constexpr int {name} = ([^;]+);", text)
        if m:
            env[name] = eval(m.group(1), {"__builtins__": {}}, env)
    return env


def _table_error(c):
    """The largest relative error of a table's entry: a weight in [2^-((b + 1) w), 2^-(b w)], bins of w
    binary orders, times 2^(kWeightBits + floor(b w)), rounded to an integer."""
    widths = np.linspace(1e-4, 37.5 * np.log2(np.e) / c["kTableBins"], 4001)[:, None]
    b = np.arange(c["kTableBins"])[None, :]
    smallest = np.exp2(c["kWeightBits"] + np.floor(b * widths) - (b + 1) * widths)
    return float((0.5 / smallest).max())


def test_draw_margin_covers_both_sums_tables():
    c = _constants()
    # Both sides of the draw's comparison are sums of table entries; besides them each has exps within
    # 8 ulp, an argument within 57 ulp and up to 64 additions.
    others = 2 * (8 + 57 + 64)
    assert c["kPickAdds"] >= 2 * _table_error(c) * 2.0 ** 53 + others


def test_table_sums_fit_their_words():
    # 2,048 entries of at most 2^kWeightBits in 52 bits beside a count of 12 (a little above: the bin of a
    # value at a bin's edge is rounded).
    c = _constants()
    assert 2048 * 2.0 ** c["kWeightBits"] * 1.01 < 2.0 ** 52
