"""A plan's compiled runs of tiny operations (tiny_rtc.cpp) against a run-time compiler that is played by a table: what a run does
when it cannot be compiled, and what becomes of the code of runs that are gone, without a device."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "dopt_amd", "csrc")

HARNESS = r"""
#include <cassert>
#include <cstdarg>
#include <memory>
#include "common.h"

static std::string error_text;
static bool broken = false, recording = false;
static int attempts = 0, launches = 0, loaded = 0, waits = 0;

extern "C" const char *dopt_hip_last_error(void) { return error_text.c_str(); }

namespace dopt {
int fail(int code, const char *fmt, ...)
{
    char buf[2048];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    error_text = buf;
    return code;
}
int rtc_load(const std::string &, int, const char *const *, hipModule_t *module, hipFunction_t *fn)
{
    attempts++;
    if (broken) return fail(DOPT_HIP_ERR_RTC, "hipRTC compilation failed");
    loaded++;
    *module = (hipModule_t)1;
    *fn = (hipFunction_t)1;
    return DOPT_HIP_OK;
}
void rtc_idle() { waits++; }
void rtc_unload(hipModule_t) { loaded--; }
bool capturing() { return recording; }
int rtc_launch(hipFunction_t, unsigned, unsigned, void **)
{
    launches++;
    return DOPT_HIP_OK;
}
}

using namespace dopt;

// out = (a + b) * a over n values
static std::unique_ptr<TinyRun> make_run(int n)
{
    std::vector<dopt_hip_tiny_node> nodes(2);
    for (int k = 0; k < 2; k++) {
        dopt_hip_tiny_node nd{};
        nd.kind = DOPT_HIP_TINY_POINTWISE;
        nd.op = k ? 2 : 0;   // mul, add
        nd.dst = 2 + k;
        nd.a = k ? 2 : 0;
        nd.b = k ? 0 : 1;
        nd.n = n;
        nodes[(size_t)k] = nd;
    }
    return std::unique_ptr<TinyRun>(new TinyRun(4, nodes));
}

static float memory[4][256];
static void *slots[4] = {memory[0], memory[1], memory[2], memory[3]};

#define CHECK(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)

int main()
{
BODY
    puts("ok");
    return 0;
}
"""


def _run(tmp_path, body):
    src, exe = os.path.join(str(tmp_path), "harness.cpp"), os.path.join(str(tmp_path), "harness")
    with open(src, "w") as f:
        f.write(HARNESS.replace("BODY", body))
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I", CSRC, "-w", "-o", exe, src,
                    os.path.join(CSRC, "tiny_rtc.cpp")], check=True)
    out = subprocess.run([exe], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout + out.stderr


def test_a_run_that_cannot_be_compiled_is_left_to_the_interpreter(tmp_path):
    _run(tmp_path, r"""
    auto run = make_run(10), other = make_run(11);
    bool done = true;
    error_text = "what an earlier call reported";
    broken = true;
    for (int i = 0; i < 3; i++) {
        CHECK(run->launch(slots, &done) == DOPT_HIP_OK);
        CHECK(!done && launches == 0 && attempts == 1);   // and is not tried again
        CHECK(error_text == "what an earlier call reported");
    }
    broken = false;
    for (int i = 0; i < 2; i++) {
        CHECK(other->launch(slots, &done) == DOPT_HIP_OK && done);
        CHECK(launches == i + 1 && attempts == 2);
    }
""")


def test_the_code_of_runs_that_are_gone_is_bounded(tmp_path):
    _run(tmp_path, r"""
    bool done;
    std::vector<std::unique_ptr<TinyRun>> live;
    for (int n = 1; n <= 200; n++) {   // a plan for every batch size
        make_run(n)->launch(slots, &done);
        CHECK(done && attempts == n && loaded == std::min(n, 64));
    }
    make_run(200)->launch(slots, &done);   // the newest are still there
    CHECK(done && attempts == 200);
    for (int n = 1; n <= 200; n++) {   // all at once: none is taken from a run that holds it
        live.push_back(make_run(n));
        live.back()->launch(slots, &done);
        live.back()->launch(slots, &done);
        CHECK(done);
    }
    CHECK(loaded >= 200 && loaded <= 264);
    auto second = make_run(7);   // shares the code of the one above
    const int before = attempts;
    second->launch(slots, &done);
    CHECK(done && attempts == before);
    recording = true;   // nothing can be waited for, so nothing is unloaded
    const int kept = loaded, waited = waits;
    for (int n = 0; n < 150; n++) live[(size_t)n].reset();
    CHECK(loaded == kept && waits == waited);
    recording = false;
    live.clear();
    CHECK(loaded <= 65 && waits > waited);
    tiny_codes_trim();
    CHECK(loaded == 1);
    second->launch(slots, &done);
    CHECK(done && attempts == before);
    tiny_codes_shutdown();   // and the run compiles its kernel again
    CHECK(loaded == 0);
    second->launch(slots, &done);
    CHECK(done && attempts == before + 1 && loaded == 1);
    second.reset();
    tiny_codes_trim();
    CHECK(loaded == 0);
""")
