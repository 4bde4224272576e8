"""Registers that inline assembly writes by name are declared: the compiler may
hold a value of its own in any other."""

from __future__ import annotations

import re
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "leanstack_amd" / "csrc"
ASM = re.compile(r'\basm\b\s*(?:volatile)?\s*\((.*?)\)\s*;', re.S)
NAMED = re.compile(r'\b(?:s_mov_b32|s_mov_b64|s_add_u32|v_mov_b32)\s+(m0|vcc|exec|s\d+|v\d+)\b')


def _statements():
    for path in sorted(CSRC.iterdir()):
        for statement in ASM.findall(path.read_text()):
            yield path.name, statement


def test_statements_are_found():
    assert any("s_mov_b32 m0" in text for _, text in _statements())


@pytest.mark.parametrize("name", sorted({name for name, _ in _statements()}))
def test_named_registers_are_clobbers(name):
    for file, text in _statements():
        if file == name:
            for register in NAMED.findall(text):
                assert f'"{register}"' in text, f"{file}: {register} is written and not declared: {text}"
