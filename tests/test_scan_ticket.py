"""The offset scan's rule for the tickets its blocks draw (fls_scan_ticket.hpp),
on the CPU: a prepared state hands out every block once, and a state that an
earlier scan has used up, that was prepared for another number of vectors, or
that no planner has prepared, gives no block a number to index by.  And the
Python side of it: a mixed_resolve without its own mixed_stats is refused before
anything is launched."""
import pathlib
import subprocess
from types import SimpleNamespace

import pytest

from fastlanesgpu_amd import selector as sel

ROOT = pathlib.Path(__file__).resolve().parents[1]

PROGRAM = r"""
#include <stdio.h>
#include <stdint.h>
#include "fls_scan_ticket.hpp"

static uint64_t s = 0x9E3779B97F4A7C15ull;
static uint64_t rnd() { s ^= s << 13; s ^= s >> 7; s ^= s << 17; return s; }
static uint32_t draw(unsigned long long& word, uint64_t n_vec, uint32_t blocks) {
    return RULE;  // as a block does: atomicAdd returns the word before the addition
}

int main() {
    const uint64_t sizes[] = {1, 2, 1023, 1024, 1025, 8195, 117188, 524289, 1048577, 1ull << 31, (1ull << 41) - 1};
    for (uint64_t n : sizes) {
        const uint32_t blocks = (uint32_t)((n + 1023) / 1024), some = blocks < 5000 ? blocks : 5000;
        unsigned long long word = fls::scan_ticket_word(n);
        for (uint32_t b = 0; b < some; ++b)
            if (draw(word, n, blocks) != b) return printf("block %u of %llu\n", b, (unsigned long long)n), 1;
        word = fls::scan_ticket_word(n) + blocks;  // used up
        for (uint32_t k = 0; k < some; ++k)
            if (draw(word, n, blocks) != fls::kNoTicket) return printf("used up, %llu\n", (unsigned long long)n), 1;
        for (uint64_t other : sizes) {
            word = fls::scan_ticket_word(other);
            if (other != n && draw(word, n, blocks) != fls::kNoTicket) return printf("other size\n"), 1;
        }
        word = fls::scan_ticket_word(n + 1);
        if (draw(word, n, blocks) != fls::kNoTicket) return printf("next size\n"), 1;
        const unsigned long long words[] = {0ull, 5ull, ~0ull, ~0ull << 32, 0xffffffffull, 1ull << 63};
        for (unsigned long long w : words) {
            word = w;
            if (draw(word, n, blocks) != fls::kNoTicket) return printf("unprepared %llx\n", w), 1;
        }
        for (int k = 0; k < 100000; ++k) {
            word = rnd();
            if (draw(word, n, blocks) != fls::kNoTicket) return printf("random\n"), 1;
        }
    }
    printf("OK\n");
    return 0;
}
"""
RULE = "fls::scan_ticket(word++, n_vec, blocks)"


def run_program(tmp_path, rule):
    src, exe = tmp_path / "ticket.cpp", tmp_path / "ticket"
    src.write_text(PROGRAM.replace("RULE", rule))
    subprocess.run(["g++", "-O2", "-std=c++17", f"-I{ROOT / 'fastlanesgpu_amd' / 'csrc'}", str(src), "-o", str(exe)],
                   check=True)
    return subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)


def test_a_ticket_is_a_block_of_this_scan_or_none(tmp_path):
    r = run_program(tmp_path, RULE)
    assert r.returncode == 0 and r.stdout.strip() == "OK", r.stdout


@pytest.mark.parametrize("rule", ["(void)n_vec, (void)blocks, (uint32_t)word++",                    # any word is a ticket
                                  "(uint32_t)(word >> 32) == fls::scan_tag(n_vec) ? (uint32_t)word++ : fls::kNoTicket",
                                  "(uint32_t)word < blocks ? (uint32_t)word++ : fls::kNoTicket"])
def test_the_check_fails_for_a_weaker_rule(tmp_path, rule):
    assert run_program(tmp_path, rule).returncode != 0


def workspace():
    return SimpleNamespace(cls=1, vmeta=2, aux=3, words=4, total=5, fallbacks=6, scratch=7, feat=8, conf=9, trial=10,
                           stats_n=None)


@pytest.mark.parametrize("between", ["nothing", "resolve", "another size", "mixed_plan", "mixed_encode",
                                     "mixed_encode_trial"])
def test_resolve_takes_its_own_statistics(monkeypatch, between):
    calls = []
    monkeypatch.setattr(sel, "call", lambda name, *a: calls.append(name))
    ws, n = workspace(), 5000
    sel.mixed_stats(16, n, ws)
    if between == "nothing":
        ws = workspace()
    elif between == "resolve":
        sel.mixed_resolve(n, ws, exhaustive=True)
    elif between != "another size":
        getattr(sel, between)(16, n, ws)
    calls.clear()
    with pytest.raises(ValueError, match="mixed_stats"):
        sel.mixed_resolve(n - (between == "another size"), ws, exhaustive=True)
    assert calls == []
    sel.mixed_stats(16, n, ws)
    sel.mixed_resolve(n, ws, exhaustive=True)
    assert calls == ["fls_mixed_stats_device", "fls_mixed_resolve_device"]
