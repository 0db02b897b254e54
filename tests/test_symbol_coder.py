"""The branch-free symbol coder of observer-less encodes against the decision by
decision range encoder, and the token CRC's four-byte steps against byte steps, both
compiled from the library's host source and run on the CPU."""
import pathlib
import shutil
import subprocess

import pytest

HOST = pathlib.Path(__file__).resolve().parent.parent / "tsac-metal_amd" / "csrc" / "host"
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

DRIVER = r"""
#include "format.hpp"
#include <cstdio>
#include <cstring>
#include <random>
using namespace tsac_hip;

static uint32_t byte_crc(const std::vector<uint16_t>& tokens)
{
    uint32_t crc = 0xffffffffu;
    for (uint32_t token : tokens)
    {
        for (int shift = 0; shift < 32; shift += 8)
        {
            crc ^= ((token >> shift) & 255) << 24;
            for (int bit = 0; bit < 8; ++bit)
            {
                crc = (crc << 1) ^ ((crc & 0x80000000u) ? 0x04c11db7u : 0u);
            }
        }
    }
    return crc;
}

int main()
{
    std::mt19937_64 random(1);
    // Splits near both ends move two bytes a decision and run up carries; extreme
    // symbols walk one edge of the interval.
    for (int kind = 0; kind < 6; ++kind)
    {
        for (int round = 0; round < 200; ++round)
        {
            const size_t count = round < 150 ? random() % 40 : 1000;
            std::vector<uint16_t> splits(count * 16), symbols(count);
            for (size_t i = 0; i < count; ++i)
            {
                symbols[i] = kind == 3 ? 1023 : kind == 4 ? 0 : random() % 1024;
                for (int level = 0; level < 10; ++level)
                {
                    const uint32_t r = uint32_t(random());
                    const uint32_t choices[6] = {1 + r % 32767, r & 1 ? 1u : 32767u, 16384, 1 + r % 40, 32767 - r % 40,
                                                 r % 3 == 0 ? 1u : r % 3 == 1 ? 32767u : 1 + r % 32767};
                    splits[i * 16 + level] = uint16_t(choices[kind]);
                }
            }
            RangeEncoder decisions(1 << 30);
            SymbolEncoder coder(count);
            for (size_t i = 0; i < count; ++i)
            {
                for (int level = 0; level < 10; ++level)
                {
                    decisions.put(splits[i * 16 + level], symbols[i] >> (9 - level) & 1);
                }
                coder.put(&splits[i * 16], symbols[i]);
            }
            if (decisions.finish() != coder.finish() || token_crc32(symbols.data(), count) != byte_crc(symbols))
            {
                std::printf("differs: kind %d round %d count %zu\n", kind, round, count);
                return 1;
            }
        }
    }
    for (uint16_t bad : {uint16_t(0), uint16_t(32768), uint16_t(65535)})
    {
        uint16_t splits[16];
        std::fill(splits, splits + 16, uint16_t(16384));
        splits[9] = bad;
        bool refused = false;
        try
        {
            SymbolEncoder(1).put(splits, 5);
        }
        catch (const Error&)
        {
            refused = true;
        }
        if (!refused)
        {
            return 2;
        }
    }
    // The coder of the largest recording by default (64 Mi symbols) touches what it writes.
    SymbolEncoder large(std::size_t(64) << 20);
    uint16_t even[16];
    std::fill(even, even + 16, uint16_t(16384));
    large.put(even, 5);
    large.finish();
    long resident = -1; // the program's own peak (getrusage's includes its parent's)
    char line[256];
    for (std::FILE* status = std::fopen("/proc/self/status", "r"); std::fgets(line, sizeof line, status);)
    {
        std::sscanf(line, "VmHWM: %ld kB", &resident);
    }
    if (resident < 0 || resident > 256 * 1024)
    {
        std::printf("%ld KiB resident\n", resident);
        return 3;
    }
    return 0;
}
"""


@pytest.mark.skipif(not pathlib.Path(HIPCC).exists(), reason="no compiler")
def test_symbol_coder_equals_the_decision_coder(tmp_path):
    (tmp_path / "driver.cpp").write_text(DRIVER)
    program = tmp_path / "driver"
    subprocess.run([HIPCC, "-O2", "-x", "c++", "-std=c++23", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    f"-I{HOST}", str(tmp_path / "driver.cpp"), str(HOST / "format.cpp"), "-o", str(program)], check=True)
    result = subprocess.run([str(program)], capture_output=True, text=True)
    assert result.returncode == 0, result.stdout
