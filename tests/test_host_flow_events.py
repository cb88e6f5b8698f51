"""Host side of fmc_flow_backward against a stand-in for the HIP runtime (its calls
are noted and nothing is launched): what may be recorded into a HIP graph
releases no event (the capture that recorded it is still open), a second call
needs no new ones, and a side stream that is the main stream needs none."""

import ctypes as C
import json
import os
import subprocess
import sys

import pytest

from flowmc_amd import _native as N

RUNTIME = r"""
#include <cstdint>
#include <cstdio>
#include <cstring>
static char notes[1 << 16];
static int n = 0, live = 0;
static void note(const char* s) { n += std::snprintf(notes + n, sizeof(notes) - n, "%s ", s); }
struct D3 { unsigned x, y, z; };
extern "C" {
const char* stand_in_notes() { return notes; }
void stand_in_clear() { n = 0; notes[0] = 0; }
int hipEventCreateWithFlags(void** e, unsigned) { *e = (void*)(intptr_t)(0x100 + ++live); note("create"); return 0; }
int hipEventDestroy(void*) { note("destroy"); return 0; }
int hipEventRecord(void*, void*) { note("record"); return 0; }
int hipStreamWaitEvent(void*, void*, unsigned) { note("wait"); return 0; }
int __hipPushCallConfiguration(D3, D3, size_t, void*) { return 0; }
int __hipPopCallConfiguration(D3*, D3*, size_t*, void**) { return 0; }
int hipLaunchKernel(const void*, D3, D3, void**, size_t, void*) { note("launch"); return 0; }
int hipFuncSetAttribute(const void*, int, int) { return 0; }
int hipGetLastError() { return 0; }
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipDeviceGetAttribute(int* v, int, int) { *v = 256; return 0; }
}
"""

CALLS = r"""
import ctypes as C, json, sys
hip = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
hip.stand_in_notes.restype = C.c_char_p
lib = C.CDLL(sys.argv[2])
P, I64, I32 = C.c_void_p, C.c_int64, C.c_int32
lib.fmc_flow_backward.argtypes = [P, P, P, P, I64] + [P] * 5 + [I64, P, P, I32, P, I32, P, I64]
lib.fmc_last_error.restype = C.c_char_p
flow = C.create_string_buffer(bytes.fromhex(sys.argv[3]))
out = []
for main, side in ((0x10, 0x20), (0x10, 0x20), (0x10, 0x10)):
    hip.stand_in_clear()
    rc = lib.fmc_flow_backward(main, side, flow, 0x1000, 64, 0x1000, 0x1000, 0x2000, 0x1000, 0x1000, 64, 0x1000, 0x1000, 2,
                               0x1000, 0, None, 0)
    out.append([rc, lib.fmc_last_error().decode() if rc else "", hip.stand_in_notes().decode().split()])
print(json.dumps(out))
"""


@pytest.fixture(scope="module")
def calls(tmp_path_factory):
    d = tmp_path_factory.mktemp("stand_in")
    (d / "hip.cpp").write_text(RUNTIME)
    (d / "calls.py").write_text(CALLS)
    subprocess.run(["g++", "-shared", "-fPIC", "-O1", "-o", str(d / "hip.so"), str(d / "hip.cpp")], check=True)
    flow = N.make_flow(5, 4, 8, [32, 32], 1, theta=0x1000, packed=0x1000, packed_bias=0x1000)
    r = subprocess.run([sys.executable, str(d / "calls.py"), str(d / "hip.so"), str(N.LIB_PATH), bytes(flow).hex()],
                       capture_output=True, text=True, timeout=120, env=dict(os.environ))
    assert r.returncode == 0, r.stderr
    got = json.loads(r.stdout.strip().splitlines()[-1])
    assert all(rc == 0 for rc, _, _ in got), got
    assert all("launch" in notes for _, _, notes in got), got  # the stand-in was called
    return [notes for _, _, notes in got]


def test_sweep_releases_no_event(calls):
    for notes in calls:
        assert "destroy" not in notes


def test_sweep_keeps_its_events(calls):
    assert calls[0].count("create") == 3
    assert "create" not in calls[1]
    assert [c for c in calls[0] if c != "create"] == calls[1]
    assert calls[1].count("record") == 2 * 4 and calls[1].count("wait") == 4 + 2 + 2


def test_sweep_on_one_stream_needs_no_events(calls):
    assert set(calls[2]) == {"launch"}
