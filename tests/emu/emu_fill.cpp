// tsm_json_masks_fill on the CPU emulation (test infrastructure) with launches
// counted and made to fail: a call that failed leaves no state behind that the
// set would take for a kept mask, and a call that copies no row makes one
// launch, its states grouped by the vocabulary's length.  Prints "ok" and exits 0 when all holds.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

static int launches = 0, fail_launch = 0, fail_record = 0, records = 0;  // fail_*: the n-th of the call, 0 none
static hipError_t last = hipSuccess;
template <class F>
static void launch(F&& f) {
    if (++launches == fail_launch) last = hipErrorInvalidValue;
    else f();
}
static hipError_t last_error() {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
static hipError_t record(hipEvent_t e, hipStream_t s) { return ++records == fail_record ? hipErrorInvalidValue : hipEventRecord(e, s); }
#define hipLaunchKernelGGL(...) launch([&] { hipLaunchKernelGGL(__VA_ARGS__); })
#define hipGetLastError last_error
#define hipEventRecord record
#include "../../tachyon_amd/csrc/tsm_mask.hip"

static int fails = 0;
#define CHECK(c, ...)                          \
    do {                                       \
        if (!(c)) {                            \
            std::fprintf(stderr, __VA_ARGS__); \
            std::fprintf(stderr, "\n");        \
            fails++;                           \
        }                                      \
    } while (0)

static tsm_json_state state_of(const char* prefix) {
    tsm_json_state s;
    tsm_json_init(&s);
    tsm_json_advance(&s, reinterpret_cast<const uint8_t*>(prefix), std::strlen(prefix));
    return s;
}

int main() {
    std::vector<uint8_t> bytes;
    std::vector<uint32_t> offsets{0}, special(10, 0u);
    for (uint32_t t = 0; t < 300; t++) {
        bytes.push_back(static_cast<uint8_t>(t));
        if (t >= 256) bytes.push_back(static_cast<uint8_t>("\"}],:0e {"[t % 9]));
        if (t >= 270) {  // tokens of text bytes only, or but for their last byte
            const std::string tail = std::string("u00e9bnf/rt00ab") + std::string(t % 40, 'x') + (t % 3 ? "" : "\"");
            bytes.resize(offsets.back());
            bytes.insert(bytes.end(), tail.begin() + t % 15, tail.end());
        }
        offsets.push_back(static_cast<uint32_t>(bytes.size()));
    }
    const tsm_vocab v{bytes.data(), offsets.data(), special.data(), 300, 0};
    const uint32_t usable = 300, nw = (usable + 31) / 32;
    const std::vector<tsm_json_state> a = {state_of("{"), state_of("{\"a\":"), state_of("{"), state_of("{\"k")};
    const std::vector<tsm_json_state> b = {state_of("{\"x\": 1"), state_of("{\"k"), state_of("{\"y\": [")};
    char err[128];
    // a call's results, or a failed one's code; counts what it launched
    auto fill = [&](tsm_json_masks* m, const std::vector<tsm_json_state>& rows, tsm_json_fill_stats* st) {
        std::vector<uint32_t> got(rows.size() * nw, 0x5A5A5A5Au), want(rows.size() * nw, 0u);
        launches = records = 0;
        const int rc = tsm_json_masks_fill(m, nullptr, &v, rows.data(), static_cast<uint32_t>(rows.size()), got.data(), nw,
                                           st, err, sizeof(err));
        fail_launch = fail_record = 0;
        if (rc != 0) return rc;
        for (size_t r = 0; r < rows.size(); r++)
            for (uint32_t t = 0; t < usable; t++)
                if (tsm_json_accepts(&rows[r], bytes.data() + offsets[t], offsets[t + 1] - offsets[t]))
                    want[r * nw + t / 32] |= 1u << (t % 32);
        CHECK(got == want, "a call's masks differ from the host automaton's");
        return rc;
    };
    // the n-th launch, and each event record, fails: with an empty set, and with one that holds some of the rows
    for (int kept = 0; kept < 2; kept++)
        for (int n = 1; n <= 4; n++) {
            tsm_json_masks* m = tsm_json_masks_create(0, 8, 8, usable, err, sizeof(err));
            tsm_json_fill_stats st;
            if (kept) CHECK(fill(m, b, &st) == 0, "fill: %s", err);
            (n <= 2 ? fail_launch : fail_record) = n <= 2 ? n : n - 2;
            const int rc = fill(m, a, &st);
            if (n > 2 || launches >= n) {  // a call of one launch has no second one to fail
                CHECK(rc != 0, "kept %d, failure %d: reported as done", kept, n);
                CHECK(n != 1 || launches == 1, "kept %d: %d launches after the first failed", kept, launches);
                CHECK(fill(m, a, &st) == 0, "fill after a failure: %s", err);
                CHECK(st.hits == 0 && st.evaluated == 3, "kept %d, failure %d: %u hits, %u evaluated after it", kept, n,
                      st.hits, st.evaluated);
            }
            tsm_json_masks_destroy(m);
        }
    {  // one launch where no row is copied: rows in new states, or a set keeping nothing
        tsm_json_masks* m = tsm_json_masks_create(0, 8, 8, usable, err, sizeof(err));
        tsm_json_masks* m0 = tsm_json_masks_create(0, 8, 0, usable, err, sizeof(err));
        tsm_json_fill_stats st;
        CHECK(fill(m, {a[0]}, &st) == 0 && launches == 1, "a new state: %d launches", launches);
        CHECK(fill(m, {a[0]}, &st) == 0 && launches == 1, "a kept state: %d launches", launches);
        CHECK(fill(m, a, &st) == 0 && launches == 2, "kept and new states: %d launches", launches);
        CHECK(fill(m0, a, &st) == 0 && launches == 1, "nothing kept: %d launches", launches);
        tsm_json_masks_destroy(m);
        tsm_json_masks_destroy(m0);
    }
    {  // states inside strings, escapes and \\u groups among them, which plain tokens leave for text
        std::vector<tsm_json_state> in;
        for (const char* p : {"{\"a", "{\"a\\", "{\"a\\u", "{\"a\\u0", "{\"a\\u00", "{\"a\\u00e", "{\"a\": \"\\", "[\"\\u12",
                              "{\"a\": [\"b\\u", "{\"a\": 1", "{\"a\": tr"})
            in.push_back(state_of(p));
        tsm_json_masks* m = tsm_json_masks_create(0, 16, 0, usable, err, sizeof(err));
        tsm_json_fill_stats st;
        CHECK(fill(m, in, &st) == 0, "fill: %s", err);
        tsm_json_masks_destroy(m);
    }
    {  // a full vocabulary's states stay together, so that equal ones meet; a short one's are spread
        using tsm::mask::states_per_group;
        for (uint32_t blocks : {392u, 501u, 594u, 1024u})
            CHECK(states_per_group(256, blocks) == 256 && states_per_group(700, blocks) == 256 && states_per_group(1, blocks) == 1,
                  "%u blocks: %u states a group", blocks, states_per_group(256, blocks));
        CHECK(states_per_group(256, 313) == 128 && states_per_group(256, 125) == 64 && states_per_group(16, 1) == 1,
              "short vocabularies: %u %u %u states a group", states_per_group(256, 313), states_per_group(256, 125),
              states_per_group(16, 1));
    }
    if (fails) return 1;
    std::printf("ok\n");
    return 0;
}
