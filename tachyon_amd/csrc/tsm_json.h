// tsm_json.h - the JSON-object constraint's byte automaton on a packed
// 12-byte state, for the host and the device alike.
//
// Tachyon's JsonObject (src/constrain.rs:88-302) is a byte-level pushdown
// automaton for one JSON object (RFC 8259): a state, a stack of open
// containers (at most 32 deep) and a count of consecutive whitespace bytes
// (at most 16).  A token is allowed when its bytes all step a copy of the
// automaton successfully (accepts_bytes, constrain.rs:280-283), it is not a
// special token and it has bytes (constrain.rs:286-290).  Here the stack is a
// 32-bit word (bit i: level i is an object), so a row's whole state fits in
// tsm_json_state and every token of the vocabulary can be probed by its own
// GPU thread from a register copy.
//
// The step below follows constrain.rs:160-277 byte for byte, including what
// Constraint::advance (constrain.rs:292-296) leaves behind after a byte the
// automaton rejects: a number's length still grows past its limit, a string
// escape still resets, and the u8 counters wrap as Rust's release build does.
#pragma once

#include <hip/hip_runtime.h>

#include "tachyon_sampler.h"

namespace tsm {
namespace json {

// tsm_json_state.state
enum : uint8_t {
    JS_VALUE = 0,        // a value must start here (the top level takes only '{')
    JS_ARRAY_START = 1,  // just after '[': a value or ']'
    JS_OBJECT_START = 2, // just after '{': a key or '}'
    JS_KEY = 3,          // after ',' in an object: a key
    JS_COLON = 4,        // after a key: ':'
    JS_AFTER = 5,        // after a value inside a container: ',' or the closing bracket
    JS_STR = 6,          // inside a string; aux = key | escape << 1 | hex << 2
    JS_NUMBER = 7,       // aux = the number's part (N_*), len = its length so far
    JS_LITERAL = 8,      // aux = the word (0 true, 1 false, 2 null), len = bytes matched
    JS_DONE = 9,         // the object is closed
};
// number parts (constrain.rs:44-54)
enum : uint8_t { N_MINUS = 0, N_ZERO, N_INT, N_DOT, N_FRAC, N_EXP, N_EXPSIGN, N_EXPDIGITS };

constexpr uint8_t kMaxWhitespace = 16;  // constrain.rs:84
constexpr uint8_t kMaxNumber = 40;      // constrain.rs:85
constexpr uint8_t kMaxDepth = 32;       // constrain.rs:86

__host__ __device__ inline void init(tsm_json_state* s) {
    s->stack = 0;
    s->depth = 0;
    s->state = JS_VALUE;
    s->aux = 0;
    s->len = 0;
    s->whitespace = 0;
    s->pad[0] = s->pad[1] = s->pad[2] = 0;
}

__host__ __device__ inline bool is_digit(uint8_t b) { return b >= '0' && b <= '9'; }
__host__ __device__ inline bool is_hex(uint8_t b) {
    return is_digit(b) || (b >= 'a' && b <= 'f') || (b >= 'A' && b <= 'F');
}
// The top container: 1 object, 0 array (depth in [1, 32]).
__host__ __device__ inline uint32_t top(const tsm_json_state& s) { return (s.stack >> ((s.depth - 1u) & 31u)) & 1u; }

__host__ __device__ inline void value_done(tsm_json_state& s) { s.state = s.depth == 0 ? JS_DONE : JS_AFTER; }

__host__ __device__ inline bool open(tsm_json_state& s, uint32_t object) {
    if (s.depth >= kMaxDepth) return false;
    s.stack = (s.stack & ((1u << s.depth) - 1u)) | (object << s.depth);
    s.depth++;
    s.state = object ? JS_OBJECT_START : JS_ARRAY_START;
    return true;
}

__host__ __device__ inline bool close(tsm_json_state& s, uint32_t object) {
    if (s.depth == 0 || top(s) != object) return false;
    s.depth--;
    value_done(s);
    return true;
}

__host__ __device__ inline bool start_value(tsm_json_state& s, uint8_t b) {
    if (s.depth == 0) return b == '{' && open(s, 1u);
    switch (b) {
        case '{': return open(s, 1u);
        case '[': return open(s, 0u);
        case '"': s.state = JS_STR; s.aux = 0; return true;
        case '-': s.state = JS_NUMBER; s.aux = N_MINUS; s.len = 1; return true;
        case '0': s.state = JS_NUMBER; s.aux = N_ZERO; s.len = 1; return true;
        case 't': s.state = JS_LITERAL; s.aux = 0; s.len = 1; return true;
        case 'f': s.state = JS_LITERAL; s.aux = 1; s.len = 1; return true;
        case 'n': s.state = JS_LITERAL; s.aux = 2; s.len = 1; return true;
        default:
            if (b >= '1' && b <= '9') {
                s.state = JS_NUMBER;
                s.aux = N_INT;
                s.len = 1;
                return true;
            }
            return false;
    }
}

// The next number part after byte b, or 0xFF when b does not continue the
// number (constrain.rs:202-213).
__host__ __device__ inline uint8_t number_next(uint8_t n, uint8_t b) {
    const bool d = is_digit(b);
    switch (n) {
        case N_MINUS: return b == '0' ? N_ZERO : (d ? N_INT : 0xFF);
        case N_ZERO: return b == '.' ? N_DOT : (b == 'e' || b == 'E') ? N_EXP : 0xFF;
        case N_INT: return b == '.' ? N_DOT : d ? N_INT : (b == 'e' || b == 'E') ? N_EXP : 0xFF;
        case N_DOT: return d ? N_FRAC : 0xFF;
        case N_FRAC: return d ? N_FRAC : (b == 'e' || b == 'E') ? N_EXP : 0xFF;
        case N_EXP: return (b == '+' || b == '-') ? N_EXPSIGN : d ? N_EXPDIGITS : 0xFF;
        case N_EXPSIGN: return d ? N_EXPDIGITS : 0xFF;
        default: return d ? N_EXPDIGITS : 0xFF;  // N_EXPDIGITS
    }
}

// Feeds one byte; false if it cannot appear here (JsonObject::step).
__host__ __device__ inline bool step(tsm_json_state& s, uint8_t b) {
    const bool ws = b == ' ' || b == '\t' || b == '\n' || b == '\r';
    if (s.state == JS_STR) {
        const uint8_t key = s.aux & 1u, esc = (s.aux >> 1) & 1u, hex = s.aux >> 2;
        if (hex > 0) {
            s.aux = static_cast<uint8_t>(key | ((hex - 1u) << 2));
            return is_hex(b);
        }
        if (esc) {
            s.aux = static_cast<uint8_t>(key | ((b == 'u' ? 4u : 0u) << 2));
            return b == '"' || b == '\\' || b == '/' || b == 'b' || b == 'f' || b == 'n' || b == 'r' || b == 't' ||
                   b == 'u';
        }
        if (b == '"') {
            if (key) s.state = JS_COLON;
            else value_done(s);
            return true;
        }
        if (b == '\\') {
            s.aux = static_cast<uint8_t>(key | 2u);
            return true;
        }
        return b >= 0x20;
    }
    if (s.state == JS_NUMBER) {
        const uint8_t next = number_next(s.aux, b);
        if (next != 0xFF) {
            const uint8_t len = s.len;
            s.aux = next;
            s.len = static_cast<uint8_t>(len + 1u);
            return len < kMaxNumber;
        }
        // the number ends here if it can; the byte then belongs to what follows
        if (!(s.aux == N_ZERO || s.aux == N_INT || s.aux == N_FRAC || s.aux == N_EXPDIGITS)) return false;
        value_done(s);
    } else if (s.state == JS_LITERAL) {
        const char* word = s.aux == 0 ? "true" : s.aux == 1 ? "false" : "null";
        const uint8_t wlen = s.aux == 1 ? 5 : 4;
        if (s.len >= wlen) return false;  // not a state step() makes: the word's end is not read past
        if (static_cast<uint8_t>(word[s.len]) != b) return false;
        if (s.len + 1u == wlen) value_done(s);
        else s.len++;
        return true;
    }
    if (ws) {
        s.whitespace = static_cast<uint8_t>(s.whitespace + 1u);
        return s.whitespace <= kMaxWhitespace && s.state != JS_DONE;
    }
    s.whitespace = 0;
    switch (s.state) {
        case JS_VALUE: return start_value(s, b);
        case JS_ARRAY_START: return b == ']' ? close(s, 0u) : start_value(s, b);
        case JS_OBJECT_START:
            if (b == '}') return close(s, 1u);
            if (b == '"') {
                s.state = JS_STR;
                s.aux = 1;  // a key
                return true;
            }
            return false;
        case JS_KEY:
            if (b == '"') {
                s.state = JS_STR;
                s.aux = 1;
                return true;
            }
            return false;
        case JS_COLON:
            if (b == ':') {
                s.state = JS_VALUE;
                return true;
            }
            return false;
        case JS_AFTER:
            if (s.depth == 0) return false;  // not reached from init(): a value inside nothing is DONE
            if (b == ',') {
                s.state = top(s) ? JS_KEY : JS_VALUE;
                return true;
            }
            if (b == '}') return close(s, 1u);
            if (b == ']') return close(s, 0u);
            return false;
        default: return false;
    }
}

// Whether these bytes may come next (JsonObject::accepts_bytes): a copy steps
// until the first byte it rejects.  Inside a string with no escape pending, a
// byte other than '"', '\\' and the control bytes only passes (step's last
// case), which is taken without the full step: a GPU wave walks its tokens in
// lockstep, and most of a string's bytes are such bytes.
__host__ __device__ inline bool accepts(tsm_json_state s, const uint8_t* bytes, uint32_t n) {
    for (uint32_t i = 0; i < n; i++) {
        const uint8_t b = bytes[i];
        if (s.state == JS_STR && s.aux <= 1u && b >= 0x20 && b != '"' && b != '\\') continue;
        if (!step(s, b)) return false;
    }
    return true;
}

// ---- the automaton as a table -----------------------------------------------
// step() with its finite part written out: a flat state per (state, aux,
// literal position), 30 byte classes, and per pair the next flat state and an
// action on the counters (stack, depth, whitespace run, number length).  A GPU
// lane then takes one table word and a few predicated operations a byte where
// step() takes a chain of data-dependent branches, which a wave of different
// tokens walks one after another.
enum : uint32_t {  // byte classes: bytes step() never tells apart
    C_CTRL = 0, C_SPACE, C_BLANK /* \t \n \r */, C_QUOTE, C_BSLASH, C_SLASH, C_LBRACE, C_RBRACE, C_LBRACK, C_RBRACK,
    C_COMMA, C_COLON, C_MINUS, C_PLUS, C_DOT, C_0, C_19, C_e, C_E, C_a, C_b, C_f, C_HEX /* c d A B C D F */, C_n,
    C_r, C_t, C_u, C_l, C_s, C_TEXT /* the rest, >= 0x20 */, C_COUNT
};
constexpr uint32_t kClasses = 32;  // table row length
static_assert(C_COUNT <= kClasses, "byte classes fit a table row");

constexpr uint32_t byte_class(uint32_t b) {
    switch (b) {
        case ' ': return C_SPACE;
        case '\t': case '\n': case '\r': return C_BLANK;
        case '"': return C_QUOTE;
        case '\\': return C_BSLASH;
        case '/': return C_SLASH;
        case '{': return C_LBRACE;
        case '}': return C_RBRACE;
        case '[': return C_LBRACK;
        case ']': return C_RBRACK;
        case ',': return C_COMMA;
        case ':': return C_COLON;
        case '-': return C_MINUS;
        case '+': return C_PLUS;
        case '.': return C_DOT;
        case '0': return C_0;
        case 'e': return C_e;
        case 'E': return C_E;
        case 'a': return C_a;
        case 'b': return C_b;
        case 'f': return C_f;
        case 'c': case 'd': case 'A': case 'B': case 'C': case 'D': case 'F': return C_HEX;
        case 'n': return C_n;
        case 'r': return C_r;
        case 't': return C_t;
        case 'u': return C_u;
        case 'l': return C_l;
        case 's': return C_s;
        default: return b >= '1' && b <= '9' ? C_19 : b < 0x20 ? C_CTRL : C_TEXT;
    }
}
// Text bytes: what passes inside a string whatever else is around.
constexpr uint32_t kTextClasses =
    ~((1u << C_CTRL) | (1u << C_BLANK) | (1u << C_QUOTE) | (1u << C_BSLASH)) & ((1u << C_COUNT) - 1u);

enum : uint32_t {  // flat states
    F_VALUE = 0, F_ARRAY_START, F_OBJECT_START, F_KEY, F_COLON, F_AFTER, F_DONE, F_ROOT /* a value at depth 0 */,
    F_STR = 8,            // + 6 * key + (0: text, 1: escape, 1 + h: h hex digits left)
    F_NUM = F_STR + 12,   // + number part
    F_LIT = F_NUM + 8,    // + kLitBase[word] + bytes matched - 1
    F_OTHER = F_LIT + 10, // none of these (not a state an accepted text leaves): stepped by step()
    F_COUNT = F_OTHER
};
// A walk keeps the containers as a shift register (the innermost in bit 0) and
// its three counters in one word, each biased so that passing its limit sets
// its top bit.
constexpr uint32_t kWsBias = 127u - kMaxWhitespace, kLenBias = 127u - kMaxNumber, kDepthBias = 127u - kMaxDepth;
constexpr uint32_t kLimits = 0x00808080u;  // whitespace, number length << 8, depth << 16
constexpr uint32_t kDepth1 = 1u << 16;

// A table entry: word x, the next flat state's row (flat * kClasses) and flags;
// word y, what is added to the counters once their low (x >> W_RESET) & 31 bits
// are cleared.
enum : uint32_t {
    W_ROW = 0x7FFu,
    W_USED = 1u << 11,     // the byte is used up (else it is taken again, after a number's end)
    W_OBJ = 1u << 12,      // a container opens or closes: an object (else an array)
    W_OPEN = 1u << 13,
    W_CLOSE = 1u << 14,
    W_END = 1u << 15,      // a value ended: what follows depends on the depth
    W_COMMA = 1u << 16,    // what follows depends on the container
    W_REJECT = 1u << 17,
    W_RESET = 18,
    W_TEXT = 1u << 23      // string text follows: a rest of text bytes only passes whole
};
struct Entry {
    uint32_t x, y;
};
constexpr Entry entry(uint32_t flat, uint32_t flags, uint32_t add = 0, uint32_t reset = 0) {
    const bool text = flat == F_STR || flat == F_STR + 6u;
    return Entry{flat * kClasses | flags | (text ? uint32_t(W_TEXT) : 0u) | reset << W_RESET, add};
}
// the steps a byte can make
constexpr Entry e_reject(uint32_t f) { return entry(f, W_REJECT | W_USED); }
constexpr Entry e_go(uint32_t next) { return entry(next, W_USED); }
constexpr Entry e_blank(uint32_t f) { return entry(f, W_USED, 1u); }
// a structural byte ends the whitespace run
constexpr Entry e_mark(uint32_t next, uint32_t flags = 0, uint32_t add = 0) {
    return entry(next, flags | W_USED, kWsBias + add, 8u);
}
constexpr Entry e_open(bool obj) {
    return obj ? e_mark(F_OBJECT_START, W_OPEN | W_OBJ, kDepth1) : e_mark(F_ARRAY_START, W_OPEN, kDepth1);
}
constexpr Entry e_close(bool obj) { return e_mark(0, W_CLOSE | W_END | (obj ? W_OBJ : 0u), 0u - kDepth1); }
constexpr Entry e_value_end() { return entry(0, W_END | W_USED); }
constexpr Entry e_number(uint32_t part) {
    return entry(F_NUM + part, W_USED, kWsBias | (kLenBias + 1u) << 8, 16u);
}
constexpr Entry e_digit(uint32_t part) { return entry(F_NUM + part, W_USED, 1u << 8); }
constexpr Entry e_number_end() { return entry(0, W_END); }

constexpr uint32_t lit_base(uint32_t word) { return word == 0 ? 0u : word == 1 ? 3u : 7u; }
constexpr uint32_t lit_class(uint32_t word, uint32_t at) {
    constexpr uint8_t w[3][5] = {{C_t, C_r, C_u, C_e, 0}, {C_f, C_a, C_l, C_s, C_e}, {C_n, C_u, C_l, C_l, 0}};
    return w[word][at];
}

// The next number part after a byte of class c, 0xFF when none (number_next).
constexpr uint32_t number_class_next(uint32_t n, uint32_t c) {
    const bool d = c == C_0 || c == C_19, ex = c == C_e || c == C_E;
    switch (n) {
        case N_MINUS: return c == C_0 ? uint32_t(N_ZERO) : (d ? uint32_t(N_INT) : 0xFFu);
        case N_ZERO: return c == C_DOT ? uint32_t(N_DOT) : ex ? uint32_t(N_EXP) : 0xFFu;
        case N_INT: return c == C_DOT ? uint32_t(N_DOT) : d ? uint32_t(N_INT) : ex ? uint32_t(N_EXP) : 0xFFu;
        case N_DOT: return d ? uint32_t(N_FRAC) : 0xFFu;
        case N_FRAC: return d ? uint32_t(N_FRAC) : ex ? uint32_t(N_EXP) : 0xFFu;
        case N_EXP: return (c == C_PLUS || c == C_MINUS) ? uint32_t(N_EXPSIGN) : d ? uint32_t(N_EXPDIGITS) : 0xFFu;
        default: return d ? uint32_t(N_EXPDIGITS) : 0xFFu;  // N_EXPSIGN, N_EXPDIGITS
    }
}

constexpr Entry table_entry(uint32_t f, uint32_t c) {
    if (f >= F_LIT) {
        const uint32_t k = f - F_LIT, word = k < 3u ? 0u : k < 7u ? 1u : 2u;
        const uint32_t at = k - lit_base(word) + 1u, n = word == 1u ? 5u : 4u;
        if (c != lit_class(word, at)) return e_reject(f);
        return at + 1u == n ? e_value_end() : e_go(f + 1u);
    }
    if (f >= F_NUM) {
        const uint32_t part = f - F_NUM, next = number_class_next(part, c);
        if (next != 0xFFu) return e_digit(next);
        const bool whole = part == N_ZERO || part == N_INT || part == N_FRAC || part == N_EXPDIGITS;
        return whole ? e_number_end() : e_reject(f);
    }
    if (f >= F_STR) {
        const uint32_t key = (f - F_STR) / 6u, sub = (f - F_STR) % 6u, text = F_STR + 6u * key;
        if (sub >= 2u) {
            const bool hex = c == C_0 || c == C_19 || c == C_a || c == C_b || c == C_e || c == C_f || c == C_E || c == C_HEX;
            return hex ? e_go(sub == 2u ? text : f - 1u) : e_reject(f);
        }
        if (sub == 1u) {
            if (c == C_u) return e_go(text + 5u);
            const bool esc = c == C_QUOTE || c == C_BSLASH || c == C_SLASH || c == C_b || c == C_f || c == C_n ||
                             c == C_r || c == C_t;
            return esc ? e_go(text) : e_reject(f);
        }
        if (c == C_QUOTE) return key ? e_go(F_COLON) : e_value_end();
        if (c == C_BSLASH) return e_go(f + 1u);
        return ((kTextClasses >> c) & 1u) ? e_go(f) : e_reject(f);
    }
    if (f == F_DONE) return e_reject(f);
    if (c == C_SPACE || c == C_BLANK) return e_blank(f);
    switch (f) {
        case F_ROOT: return c == C_LBRACE ? e_open(true) : e_reject(f);
        case F_OBJECT_START:
            if (c == C_RBRACE) return e_close(true);
            return c == C_QUOTE ? e_mark(F_STR + 6u) : e_reject(f);
        case F_KEY: return c == C_QUOTE ? e_mark(F_STR + 6u) : e_reject(f);
        case F_COLON: return c == C_COLON ? e_mark(F_VALUE) : e_reject(f);
        case F_AFTER:
            if (c == C_COMMA) return e_mark(F_VALUE, W_COMMA);
            if (c == C_RBRACE) return e_close(true);
            return c == C_RBRACK ? e_close(false) : e_reject(f);
        default: break;  // F_VALUE, F_ARRAY_START
    }
    if (f == F_ARRAY_START && c == C_RBRACK) return e_close(false);
    switch (c) {
        case C_LBRACE: return e_open(true);
        case C_LBRACK: return e_open(false);
        case C_QUOTE: return e_mark(F_STR);
        case C_MINUS: return e_number(N_MINUS);
        case C_0: return e_number(N_ZERO);
        case C_19: return e_number(N_INT);
        case C_t: return e_mark(F_LIT + lit_base(0));
        case C_f: return e_mark(F_LIT + lit_base(1));
        case C_n: return e_mark(F_LIT + lit_base(2));
        default: return e_reject(f);
    }
}

constexpr uint32_t kNotText = 0x80u;

struct Tables {
    Entry next[F_COUNT * kClasses];
    // per flat state: the classes a token may start with (F_OTHER: all); a
    // number that can end hands the byte to what follows a value
    uint32_t first[F_COUNT + 1];
    uint8_t cls[256];  // a byte's class, with kNotText
};
constexpr Tables make_tables() {
    Tables t{};
    for (uint32_t f = 0; f < F_COUNT; f++)
        for (uint32_t c = 0; c < kClasses; c++) {
            const Entry e = c < C_COUNT ? table_entry(f, c) : e_reject(f);
            t.next[f * kClasses + c] = e;
            if (!(((e.x & W_USED) ? e : table_entry(F_AFTER, c)).x & W_REJECT)) t.first[f] |= 1u << c;
        }
    t.first[F_OTHER] = 0xFFFFFFFFu;
    for (uint32_t b = 0; b < 256u; b++) t.cls[b] = static_cast<uint8_t>(byte_class(b) | (((kTextClasses >> byte_class(b)) & 1u) ? 0u : kNotText));
    return t;
}

// A state's flat state.
__host__ __device__ inline uint32_t flat_of(const tsm_json_state& s) {
    if (s.depth > kMaxDepth || s.whitespace > kMaxWhitespace) return F_OTHER;
    switch (s.state) {
        case JS_VALUE: return s.depth ? uint32_t(F_VALUE) : uint32_t(F_ROOT);
        case JS_DONE: return F_DONE;
        case JS_STR: {
            const uint32_t key = s.aux & 1u, esc = (s.aux >> 1) & 1u, hex = s.aux >> 2;
            if (hex > 4u || (hex && esc) || (key && s.depth == 0)) return F_OTHER;
            return F_STR + 6u * key + (hex ? 1u + hex : esc);
        }
        case JS_NUMBER: return s.aux <= N_EXPDIGITS && s.len <= kMaxNumber ? F_NUM + s.aux : uint32_t(F_OTHER);
        case JS_LITERAL:
            if (s.aux > 2u || s.len == 0 || s.len >= (s.aux == 1u ? 5u : 4u)) return F_OTHER;
            return F_LIT + lit_base(s.aux) + s.len - 1u;
        default:
            if (s.depth == 0 || s.state > JS_DONE) return F_OTHER;
            return s.state;  // JS_ARRAY_START .. JS_AFTER: the flat states have the same numbers
    }
}
static_assert(int(F_ARRAY_START) == int(JS_ARRAY_START) && int(F_OBJECT_START) == int(JS_OBJECT_START) &&
                  int(F_KEY) == int(JS_KEY) && int(F_COLON) == int(JS_COLON) && int(F_AFTER) == int(JS_AFTER),
              "structural states keep their numbers");

// A state with flat state f without what no later byte can depend on: aux and
// len outside strings, numbers and literals (what they left behind), stack
// levels above the depth, everything of a closed object.
__host__ __device__ inline void forget(tsm_json_state* s, uint32_t f) {
    s->pad[0] = s->pad[1] = s->pad[2] = 0;
    if (f == F_OTHER) return;
    if (f < F_STR) s->aux = 0;
    if (f < F_NUM) s->len = 0;
    s->stack &= s->depth < kMaxDepth ? (1u << s->depth) - 1u : 0xFFFFFFFFu;
    if (f == F_DONE) {
        s->stack = 0;
        s->depth = s->whitespace = 0;
    }
}

// A walk through a token's byte classes.
struct Walk {
    uint32_t row, stack, count;
};
__host__ __device__ inline Walk walk_of(const tsm_json_state& s, uint32_t f) {
    Walk w{f * kClasses, 0u, (s.whitespace + kWsBias) | (f >= F_NUM && f < F_LIT ? s.len + kLenBias : 0u) << 8 |
                                 (s.depth + kDepthBias) << 16};
    for (uint32_t i = 0; i < s.depth; i++) w.stack = w.stack << 1 | ((s.stack >> i) & 1u);
    return w;
}
// One step by table entry e = next[row + (class & 31)]; false when the byte is
// rejected.  (A container closes only inside one: at depth 0 no flat state has
// a closing step.)
__host__ __device__ inline bool step_entry(Walk& w, Entry e) {
    const uint32_t obj = (e.x / W_OBJ) & 1u, top = w.stack & 1u;
    bool bad = (e.x & W_REJECT) != 0u;
    bad |= (e.x & W_CLOSE) && top != obj;
    w.count = (w.count & (0xFFFFFFFFu << ((e.x >> W_RESET) & 31u))) + e.y;
    bad |= (w.count & kLimits) != 0u;
    w.stack = (e.x & W_OPEN) ? w.stack << 1 | obj : (e.x & W_CLOSE) ? w.stack >> 1 : w.stack;
    uint32_t row = e.x & W_ROW;
    if (e.x & W_END) row = (w.count >> 16) == kDepthBias ? F_DONE * kClasses : F_AFTER * kClasses;
    if ((e.x & W_COMMA) && top) row = F_KEY * kClasses;
    w.row = row;
    return !bad;
}

}  // namespace json
}  // namespace tsm
