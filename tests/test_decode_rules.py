"""The host rules of the one-launch decode step (async-gpu_amd/csrc/decode_rules.h), compiled by themselves: no GPU."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    """A program that evaluates the expressions on its standard input's lines: `bytes d ff layers vocab int4`,
    `pays groups d heads batch ctx`, `touches MB batch groups - -`."""
    d = tmp_path_factory.mktemp("rules")
    src, exe = d / "rules.cpp", d / "rules"
    src.write_text('''
#include <cstdio>
#include <cstring>
#include "decode_rules.h"
int main() {
    char what[16];
    int a[5];
    while (std::scanf("%15s %d %d %d %d %d", what, a, a + 1, a + 2, a + 3, a + 4) == 6)
        if (!std::strcmp(what, "bytes")) std::printf("%.0f\\n", pk_token_bytes(a[0], a[1], a[2], a[3], a[4]));
        else if (!std::strcmp(what, "touches")) std::printf("%d\\n", (int)pk_touches_ahead(1e6 * a[0], a[1], a[2]));
        else std::printf("%d\\n", (int)pk_pays_rule(a[0], a[1], a[2], a[3], a[4]));
    return 0;
}
''')
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I", os.path.join(ROOT, "async-gpu_amd", "csrc"), str(src), "-o", str(exe)], check=True)

    def ask(lines):
        r = subprocess.run([str(exe)], input="\n".join(lines), capture_output=True, text=True, timeout=60, check=True)
        return [float(x) for x in r.stdout.split()]

    return ask


def test_bytes_of_a_token_weigh_the_head_by_its_type(rules):
    """0.625 bytes per int4 weight with its scale, 4 per fp32 one; whether the head is in the launch or follows it is no matter.  12 x 768
    with an int4 head is 77 MB for any number of sequences (below the 200 MB from which the weights are touched ahead), with an
    fp32 head 207 MB."""
    d, ff, layers, vocab = 768, 3072, 12, 50257
    int4, f32 = rules([f"bytes {d} {ff} {layers} {vocab} 1", f"bytes {d} {ff} {layers} {vocab} 0"])
    block = (4 * d * d + 2 * d * ff) * layers
    assert int4 == pytest.approx(0.625 * (block + d * vocab), abs=1)
    assert f32 == pytest.approx(0.625 * block + 4 * d * vocab, abs=1)
    assert int4 < 200e6 < f32


@pytest.mark.parametrize("groups,d,heads", [(4, 64, 1), (4, 192, 3), (4, 256, 4), (4, 768, 12), (2, 1024, 16), (2, 1280, 20), (1, 1600, 25), (1, 1920, 30)])
def test_one_launch_pays_less_with_more_sequences_and_longer_contexts(rules, groups, d, heads):
    """Once a launch per stage is the faster step it stays so for more sequences and for a longer context: the line has no islands.
    Three sequences of a 1600-wide model, where the Linear workgroups take every stage, are slower as one launch whatever the
    context (24 x 1600, ms per step, one launch / per stage: 0.98 / 0.93 at 64 cached positions, 1.05 / 1.02 at 300, 1.30 / 1.25 at 900); two
    are always faster."""
    ctxs = range(1, 1025)
    pays = {b: rules([f"pays {groups} {d} {heads} {b} {c}" for c in ctxs]) for b in range(2, 9)}
    for b, p in pays.items():
        assert set(p) <= {0.0, 1.0} and sorted(p, reverse=True) == p
        if b > 2:
            assert all(x <= y for x, y in zip(p, pays[b - 1]))
    assert all(pays[2])
    if groups == 4:  # up to 256 keys whatever the width (12 x 256, eight sequences: 0.23 / 0.28)
        assert all(pays[8][:256])
    if d == 1600:
        assert not any(pays[3])


def test_weights_are_touched_ahead_for_large_models_and_few_groups(rules):
    """One sequence: by size; several: with one or two groups of Linear workgroups whatever the size, with four by size."""
    ask = lambda mb, batch, groups: bool(rules([f"touches {mb} {batch} {groups} 0 0"])[0])
    assert not ask(77, 1, 2) and not ask(161, 1, 2) and ask(221, 1, 2)
    assert ask(77, 2, 2) and ask(20, 3, 1) and not ask(77, 4, 4) and ask(221, 4, 4)
