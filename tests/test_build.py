"""What the build leaves out when the compiler does not know it (vesin_amd/_build.py), with stand-ins for the compiler."""

import os
import stat

import pytest

from vesin_amd import _build


def _compiler(folder, refused):
    """A compiler that accepts every source that does not hold `refused`, and every flag but that."""
    path = folder / "hipcc"
    path.write_text(f'#!/bin/sh\nfor a in "$@"; do case "$a" in *{refused}*) exit 1;; *.hip) ! grep -q "{refused}" "$a" || exit 1;; esac; done\n')
    os.chmod(path, stat.S_IRWXU)
    return str(path)


@pytest.mark.parametrize("refused", ["nothing", "writelane", "max-regs"])
def test_what_the_compiler_does_not_know_is_left_out(refused, tmp_path):
    flags = _build.accepted_flags(_compiler(tmp_path, refused))
    assert ("-DVESIN_HIP_NO_WRITE_LANE" in flags) == (refused == "writelane")
    assert any("max-regs" in flag for flag in flags) == (refused != "max-regs")
    assert all(flag in flags for flag in _build.FLAGS)
