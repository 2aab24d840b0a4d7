// The mask producer's table and kernel on the CPU emulation (test
// infrastructure): every step of the table against json::step() over random
// states and tokens, and tsm_json_mask's words against the host stepping for
// batches past one workgroup's states and tokens past its stage.  Prints "ok"
// and exits 0 when all agree.
#include "../../tachyon_amd/csrc/tsm_mask.hip"

#include <cstdio>
#include <random>
#include <string>
#include <vector>

using namespace tsm::json;

static std::mt19937 rng(7);
static uint32_t pick(uint32_t n) { return static_cast<uint32_t>(rng() % n); }
static const std::string kJsonBytes = "{}[]\",:0123456789.eE+- \\utrufalsn\n\tbdFxa/";
static uint8_t any_byte() { return pick(20) ? static_cast<uint8_t>(kJsonBytes[pick(kJsonBytes.size())]) : static_cast<uint8_t>(pick(256)); }

// A state some text leaves, now and then one that only rejected bytes, or no
// text at all, can leave.
static tsm_json_state random_state() {
    tsm_json_state s;
    init(&s);
    if (pick(8)) (void)step(s, '{');
    for (uint32_t i = pick(24); i > 0; i--) {
        tsm_json_state c = s;
        if (step(c, any_byte()) || pick(6) == 0) s = c;
    }
    if (pick(20) == 0) s.whitespace = static_cast<uint8_t>(pick(20));
    if (pick(20) == 0) s.len = static_cast<uint8_t>(pick(64));
    if (pick(30) == 0) {
        s.depth = static_cast<uint8_t>(pick(34));
        s.stack = rng();
    }
    if (pick(100) == 0) {
        s.state = static_cast<uint8_t>(pick(12));
        s.aux = static_cast<uint8_t>(pick(24));
    }
    return s;
}
// A token that state s accepts for as long as chance allows, or any bytes.
static std::string random_token(const tsm_json_state& s) {
    std::string t;
    tsm_json_state c = s;
    const bool fit = pick(2);
    for (uint32_t i = 1 + pick(pick(4) ? 6 : 40); i > 0; i--) {
        uint8_t b = any_byte();
        for (int k = 0; fit && k < 30; k++, b = any_byte()) {
            tsm_json_state d = c;
            if (step(d, b)) break;
        }
        (void)step(c, b);
        t.push_back(static_cast<char>(b));
    }
    return t;
}

static int table_against_step() {
    static constexpr Tables tab = make_tables();
    for (long it = 0; it < 300000; it++) {
        tsm_json_state s = random_state();
        const std::string t = random_token(s);
        const uint8_t* b = reinterpret_cast<const uint8_t*>(t.data());
        const bool want = accepts(s, b, static_cast<uint32_t>(t.size()));
        const uint32_t f = flat_of(s);
        if (f == F_OTHER) continue;
        forget(&s, f);
        Walk w = walk_of(s, f);
        bool got = true;
        for (size_t i = 0; got && i < t.size();) {
            const Entry e = tab.next[w.row + (tab.cls[b[i]] & (kClasses - 1u))];
            got = step_entry(w, e);
            i += (e.x / W_USED) & 1u;
        }
        const bool starts = (tab.first[f] >> (tab.cls[b[0]] & (kClasses - 1u))) & 1u;
        if (got != want || (want && !starts)) {
            std::fprintf(stderr, "state %u aux %u len %u depth %u ws %u: step %d table %d starts %d\n", s.state, s.aux,
                         s.len, s.depth, s.whitespace, want, got, starts);
            return 1;
        }
    }
    return 0;
}

static int masks_against_step(uint32_t rows, bool long_tokens) {
    std::vector<uint8_t> bytes;
    std::vector<uint32_t> offsets{0};
    for (uint32_t i = 0; i < 600; i++) {
        std::string t = i < 256 ? std::string(1, static_cast<char>(i)) : random_token(random_state());
        if (i % 97 == 0) t.clear();
        if (long_tokens && i >= 256 && i < 512) t = std::string("\"") + std::string(80, 'x') + (i & 1 ? "\"" : "");
        bytes.insert(bytes.end(), t.begin(), t.end());
        offsets.push_back(static_cast<uint32_t>(bytes.size()));
    }
    std::vector<uint32_t> special(19, 0u);
    special[3] = 0x00010010u;
    const uint32_t n = 600, usable = 611, nw = (usable + 31) / 32, stride = nw + 1;
    const tsm_vocab v{bytes.data(), offsets.data(), special.data(), n, 0};
    std::vector<tsm_json_state> st;
    for (uint32_t r = 0; r < rows; r++) st.push_back(r > 2 && pick(2) ? st[pick(r)] : random_state());
    std::vector<uint32_t> got(static_cast<size_t>(rows) * stride, 0x5A5A5A5Au);
    char err[128];
    if (tsm_json_mask(nullptr, &v, st.data(), rows, usable, got.data(), stride, err, sizeof(err)) != 0) {
        std::fprintf(stderr, "tsm_json_mask: %s\n", err);
        return 1;
    }
    for (uint32_t r = 0; r < rows; r++) {
        for (uint32_t w = 0; w < nw; w++) {
            uint32_t want = 0;
            for (uint32_t t = 32 * w; t < 32 * w + 32 && t < n; t++) {
                const uint32_t len = offsets[t + 1] - offsets[t];
                if (!len || ((special[t >> 5] >> (t & 31u)) & 1u)) continue;
                if (accepts(st[r], bytes.data() + offsets[t], len)) want |= 1u << (t & 31u);
            }
            if (got[static_cast<size_t>(r) * stride + w] != want) {
                std::fprintf(stderr, "rows %u row %u word %u: %08x, want %08x\n", rows, r, w, got[r * stride + w], want);
                return 1;
            }
        }
        if (got[static_cast<size_t>(r) * stride + nw] != 0x5A5A5A5Au) return 1;
    }
    return 0;
}

int main() {
    if (table_against_step()) return 1;
    if (masks_against_step(3, false) || masks_against_step(300, true)) return 1;
    std::printf("ok\n");
    return 0;
}
