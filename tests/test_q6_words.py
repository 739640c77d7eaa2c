"""The rule by which the exact linear reads Q6_K blocks from whole words (csrc/q6_words.hpp), compiled for the host."""
import ctypes
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "neuralfn_amd" / "csrc"
BLOCK_BYTES, REACH = 210, 196  # a block, and how far from the word at or before it the pieces of its codes reach


@pytest.fixture(scope="module")
def past_word(tmp_path_factory):
    folder = tmp_path_factory.mktemp("q6_words")
    source, library = folder / "rule.cpp", folder / "rule.so"
    source.write_text('#include "q6_words.hpp"\n'
                      'extern "C" std::uint32_t past_word(std::uintptr_t t, std::uintptr_t b) { return nfn::q6_past_word(t, b); }\n')
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", f"-I{CSRC}", str(source), "-o", str(library)], check=True)
    call = ctypes.CDLL(str(library)).past_word
    call.argtypes, call.restype = [ctypes.c_size_t, ctypes.c_size_t], ctypes.c_uint32
    return call


@pytest.mark.parametrize("offset", [0, 1, 2, 3])
@pytest.mark.parametrize("rows,blocks", [(1, 1), (1, 2), (3, 3), (2, 8)])
def test_pieces_of_a_block_stay_inside_the_tensor(past_word, offset, rows, blocks):
    tensor = (1 << 40) + offset
    end = tensor + rows * blocks * BLOCK_BYTES
    for index in range(rows * blocks):
        block = tensor + index * BLOCK_BYTES
        start = block - past_word(tensor, block)
        assert tensor <= start <= block and start + REACH <= end
        if offset == 0:
            assert start % 4 == 0
