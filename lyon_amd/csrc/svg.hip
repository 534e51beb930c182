// SVG path data on the device: lyon_extra's PathParser (crates/extra/src/parser.rs:140-462)
// writing into lyon_path's Path layout (BuilderImpl, crates/path/src/path.rs:516-611).  The
// parse is a serial state machine over the characters; a wave per string finds the numbers
// and commands of a well-formed one in parallel, and a lane walks each string that is not, or
// that uses what the wave does not handle.  Both write into a staging room sized by the
// string's length; scans of the counts place the paths end to end and a copy kernel moves
// them there.
//
// Numbers: the parser collects `-? digits* (. digits*)? ([eE] -? digits*)?` and converts it
// with Rust's `str::parse::<f32>`, which is correctly rounded (round half to even) for
// every input.  Here: up to 19 significant digits are kept in a u64 (more set a sticky
// bit); when they fit 2^53 and the decimal exponent is within ±22, one IEEE double
// operation gives the value correctly rounded to double, and its rounding to f32 is the
// correct one unless the double lies exactly on an f32 midpoint; every other case is
// rounded exactly with 320-bit integer arithmetic, longer digit strings by comparing their
// remaining digits with the decimal expansion of the midpoint they straddle.
//
// Arcs: SvgArc::to_arc (Arc::from_svg_arc, crates/geom/src/arc.rs:58-146) and
// Arc::for_each_quadratic_bezier_with_t (arc.rs:668-701), as the parser does
// (parser.rs:287-315).  Only ASCII input is accepted: a non-ASCII byte reached by the
// parser ends the path with the NonAscii error.
#include <hip/hip_runtime.h>

#include "arc_core.h"
#include "lyg_math.h"
#include "lyg_types.h"
#include "wave.h"

namespace lyg {

namespace {

// ---- decimal to f32 -------------------------------------------------------------------
constexpr int BW = 10;  // 320-bit unsigned integers, little-endian 32-bit words
struct Big {
    uint32_t w[BW];
};

__device__ void big_set(Big& b, uint64_t v) {
#pragma unroll
    for (int i = 0; i < BW; ++i) b.w[i] = 0;
    b.w[0] = (uint32_t)v;
    b.w[1] = (uint32_t)(v >> 32);
}
__device__ void big_mul(Big& b, uint32_t m) {
    uint64_t c = 0;
#pragma unroll
    for (int i = 0; i < BW; ++i) {
        const uint64_t t = (uint64_t)b.w[i] * m + c;
        b.w[i] = (uint32_t)t;
        c = t >> 32;
    }
}
__device__ void big_pow10(Big& b, int e) {
    const uint32_t P[9] = {1u, 10u, 100u, 1000u, 10000u, 100000u, 1000000u, 10000000u,
                           100000000u};
    while (e >= 9) {
        big_mul(b, 1000000000u);
        e -= 9;
    }
    if (e > 0) big_mul(b, P[e]);
}
__device__ void big_shl(Big& b, int s) {
    const int ws = s >> 5, bs = s & 31;
    for (int i = BW - 1; i >= 0; --i) {
        const int j = i - ws;
        const uint32_t hi = j >= 0 ? b.w[j] : 0u;
        const uint32_t lo = j - 1 >= 0 ? b.w[j - 1] : 0u;
        b.w[i] = bs ? (hi << bs) | (lo >> (32 - bs)) : hi;
    }
}
__device__ int big_cmp(const Big& a, const Big& b) {
    for (int i = BW - 1; i >= 0; --i)
        if (a.w[i] != b.w[i]) return a.w[i] < b.w[i] ? -1 : 1;
    return 0;
}
__device__ void big_sub(Big& a, const Big& b) {
    int64_t br = 0;
#pragma unroll
    for (int i = 0; i < BW; ++i) {
        int64_t t = (int64_t)a.w[i] - (int64_t)b.w[i] - br;
        br = t < 0 ? 1 : 0;
        a.w[i] = (uint32_t)(t + (br << 32));
    }
}
__device__ int big_bits(const Big& a) {
    for (int i = BW - 1; i >= 0; --i)
        if (a.w[i]) return 32 * i + 32 - __builtin_clz(a.w[i]);
    return 0;
}

// f32 bits of w * 10^e correctly rounded; sticky +1 / -1 says the exact value lies just
// above / below w * 10^e (it only breaks ties).  Needs w > 0 and the value within
// [10^-46, 10^39].
__device__ uint32_t exact_round(uint64_t w, int e, int sticky) {
    Big N, D;
    big_set(N, w);
    big_set(D, 1);
    if (e >= 0) big_pow10(N, e);
    else big_pow10(D, -e);
    int k = big_bits(N) - big_bits(D);  // N / D in (2^(k-1), 2^(k+1))
    {
        Big a = N, b = D;
        if (k >= 0) big_shl(b, k);
        else big_shl(a, -k);
        if (big_cmp(a, b) < 0) --k;  // now 2^k <= N / D < 2^(k+1)
    }
    if (k > 127) return 0x7f800000u;
    const int s = k >= -126 ? 23 - k : 149;
    if (s >= 0) big_shl(N, s);
    else big_shl(D, -s);
    uint32_t q = 0;  // floor(N / D) < 2^24
    for (int bit = 24; bit >= 0; --bit) {
        Big t = D;
        big_shl(t, bit);
        if (big_cmp(N, t) >= 0) {
            big_sub(N, t);
            q |= 1u << bit;
        }
    }
    big_shl(N, 1);  // 2 * remainder against D
    int c = big_cmp(N, D);
    if (c == 0) c = sticky != 0 ? sticky : ((q & 1u) ? 1 : -1);
    if (c > 0) ++q;
    if (k >= -126) {
        if (q == (1u << 24)) {
            q = 1u << 23;
            ++k;
        }
        if (k > 127) return 0x7f800000u;
        return ((uint32_t)(k + 127) << 23) | (q - (1u << 23));
    }
    return q;  // subnormal; q == 2^23 is the smallest normal number
}

// w * 10^e through one double operation (w <= 2^53, |e| <= 22: both operands exact, so the
// double is correctly rounded); false when the double is an f32 midpoint.
__device__ bool fast_round(uint64_t w, int e, uint32_t* bits) {
    if (w > (1ull << 53) || e < -22 || e > 22) return false;
    double p = 1.0;
    for (int i = 0; i < (e < 0 ? -e : e); ++i) p *= 10.0;  // exact up to 10^22
    const double d = e >= 0 ? (double)w * p : (double)w / p;
    const float lo = __double2float_rz(d);
    const double dl = (double)lo;
    if (dl == d) {
        *bits = __float_as_uint(lo);
        return true;
    }
    const uint32_t hb = __float_as_uint(lo) + 1u;
    const double mid = (dl + (double)__uint_as_float(hb)) * 0.5;
    if (d == mid) return false;
    *bits = d < mid ? __float_as_uint(lo) : hb;
    return true;
}

__device__ __forceinline__ bool is_digit(uint32_t c) { return c >= '0' && c <= '9'; }

// Beyond 19 significant digits, when w * 10^e and (w + 1) * 10^e round to different f32
// values lo and hi (then adjacent: the interval is 1e-18 of the value wide), the value
// rounds by where it lies against their midpoint m = mm * 2^q.  With r = m / 10^e - w in
// (0, 1) as the fraction rn / rd, the remaining digits d20 d21 ... (the fraction 0.d20d21...
// of the value over 10^e) are compared with r's decimal digits one at a time; r is dyadic
// over a power of ten, so its expansion ends.  Returns lo or hi (ties to even).
__device__ uint32_t decide_midpoint(const uint8_t* s, uint32_t a, uint32_t b, uint64_t w, int e,
                                    uint32_t lo) {
    uint64_t mm;
    int q;
    if ((lo >> 23) == 0) {  // zero or subnormal: lo * 2^-149, the midpoint (2 lo + 1) 2^-150
        mm = 2ull * lo + 1;
        q = -150;
    } else {
        mm = 2ull * ((lo & 0x7fffffu) | 0x800000u) + 1;
        q = (int)(lo >> 23) - 151;
    }
    // r = mm * 2^q * 10^-e - w = rn / rd, rd = 2^max(-q, 0) * 10^max(e, 0)
    Big rn, rd, t;
    big_set(rn, mm);
    if (q > 0) big_shl(rn, q);
    if (e < 0) big_pow10(rn, -e);
    big_set(rd, 1);
    if (q < 0) big_shl(rd, -q);
    if (e > 0) big_pow10(rd, e);
    t = rd;
    big_mul(t, (uint32_t)(w >> 32));
    big_shl(t, 32);
    {
        Big u = rd;
        big_mul(u, (uint32_t)w);
        // t += u
        uint64_t c = 0;
        for (int i = 0; i < BW; ++i) {
            const uint64_t v = (uint64_t)t.w[i] + u.w[i] + c;
            t.w[i] = (uint32_t)v;
            c = v >> 32;
        }
    }
    big_sub(rn, t);  // w * rd <= m * rd / 10^e: no borrow
    // the digits after the 19th significant one, in order
    int sig = 0;
    for (uint32_t i = a; i < b; ++i) {
        const uint32_t ch = s[i];
        if (ch == 'e' || ch == 'E') break;
        if (!is_digit(ch)) continue;
        const uint32_t d = ch - '0';
        if (sig == 0 && d == 0) continue;  // leading zeros
        if (++sig <= 19) continue;
        big_mul(rn, 10);  // next digit of r: floor(10 rn / rd), at most 9
        uint32_t dm = 0;
        while (big_cmp(rn, rd) >= 0) {
            big_sub(rn, rd);
            ++dm;
        }
        if (d != dm) return d > dm ? lo + 1 : lo;
    }
    bool zero = true;
    for (int i = 0; i < BW; ++i) zero = zero && rn.w[i] == 0;
    if (!zero) return lo;          // the digits end below m
    return (lo & 1u) ? lo + 1 : lo;  // exactly m: to even
}

enum { NUM_OK = 0, NUM_SYNTAX = 1 };

// str::parse::<f32> of s[a, b), which holds what the parser collected.
__device__ int parse_f32(const uint8_t* s, uint32_t a, uint32_t b, float* out) {
    uint32_t i = a;
    bool neg = false;
    if (i < b && s[i] == '-') {
        neg = true;
        ++i;
    }
    uint64_t w = 0;
    int kept = 0, mant = 0;
    int64_t shift = 0;  // decimal exponent contributed by the digits
    bool sticky = false;
    while (i < b && is_digit(s[i])) {
        const uint32_t d = s[i] - '0';
        ++mant;
        if (kept == 0 && d == 0) {
        } else if (kept < 19) {
            w = w * 10 + d;
            ++kept;
        } else {
            ++shift;
            sticky |= d != 0;
        }
        ++i;
    }
    if (i < b && s[i] == '.') {
        ++i;
        while (i < b && is_digit(s[i])) {
            const uint32_t d = s[i] - '0';
            ++mant;
            if (kept == 0 && d == 0) {
                --shift;
            } else if (kept < 19) {
                w = w * 10 + d;
                ++kept;
                --shift;
            } else {
                sticky |= d != 0;
            }
            ++i;
        }
    }
    if (mant == 0) return NUM_SYNTAX;
    int64_t ex = 0;
    if (i < b && (s[i] == 'e' || s[i] == 'E')) {
        ++i;
        bool eneg = false;
        if (i < b && s[i] == '-') {
            eneg = true;
            ++i;
        }
        int ed = 0;
        while (i < b && is_digit(s[i])) {
            ex = ex * 10 + (s[i] - '0');
            if (ex > 1000000) ex = 1000000;
            ++ed;
            ++i;
        }
        if (ed == 0) return NUM_SYNTAX;
        if (eneg) ex = -ex;
    }
    if (i != b) return NUM_SYNTAX;
    uint32_t bits;
    const int64_t e64 = ex + shift;
    if (w == 0 || e64 + kept <= -46) {
        bits = 0;
    } else if (e64 + kept > 39) {
        bits = 0x7f800000u;
    } else {
        const int e = (int)e64;
        if (sticky) {
            const uint32_t lo = exact_round(w, e, 1);
            const uint32_t hi = exact_round(w + 1, e, -1);
            bits = lo == hi ? lo : decide_midpoint(s, a, b, w, e, lo);
        } else if (!fast_round(w, e, &bits)) {
            bits = exact_round(w, e, 0);
        }
    }
    *out = __uint_as_float(bits | (neg ? 0x80000000u : 0u));
    return NUM_OK;
}

// ---- the character source (parser.rs:48-126) ------------------------------------------
struct Src {
    const uint8_t* s;
    uint32_t pos, end;  // next byte to read, end of the string
    uint32_t at;        // byte index of `cur` (end once finished)
    uint32_t cur;
    int line, col;
    bool finished;
    bool non_ascii;
    int na_line, na_col;
};

__device__ void src_take(Src& S, uint32_t c) {
    if (c >= 0x80u && !S.non_ascii) {
        S.non_ascii = true;
        S.na_line = S.line;
        S.na_col = S.col;
    }
    S.cur = c;
}
__device__ void src_init(Src& S, const uint8_t* s, uint32_t a, uint32_t b) {
    S.s = s;
    S.end = b;
    S.non_ascii = false;
    S.na_line = S.na_col = 0;
    S.line = 0;
    S.col = 0;
    if (a < b) {
        S.at = a;
        S.pos = a + 1;
        S.finished = false;
        src_take(S, s[a]);
        if (S.cur == '\n') S.line = 1;
    } else {
        S.at = b;
        S.pos = b;
        S.cur = ' ';
        S.finished = true;
    }
}
__device__ void src_advance(Src& S) {
    if (S.finished) return;
    if (S.pos < S.end) {
        const uint32_t c = S.s[S.pos];
        S.at = S.pos;
        ++S.pos;
        if (c == '\n') {
            S.cur = '\n';
            ++S.line;
            S.col = -1;
        } else {
            ++S.col;
            src_take(S, c);
        }
    } else {
        S.cur = '~';
        S.finished = true;
        S.at = S.end;
    }
}
__device__ __forceinline__ bool is_ws(uint32_t c) { return c == ' ' || (c >= 9 && c <= 13); }
__device__ void skip_ws(Src& S) {
    while (!S.finished && (is_ws(S.cur) || S.cur == ',')) src_advance(S);
}

// ---- the output: BuilderImpl (path.rs:516-611) ----------------------------------------
template <bool EMIT>
struct Out {
    uint8_t* verbs;
    float2* points;
    uint32_t nv, np;
    vec2 first;
    uint32_t cap_v, cap_p;  // staging room of the string (writes beyond it are dropped)
    __device__ void pt(vec2 p) {
        if (EMIT && np < cap_p) points[np] = make_float2(p.x, p.y);
        ++np;
    }
    __device__ void verb(uint32_t v) {
        if (EMIT && nv < cap_v) verbs[nv] = (uint8_t)v;
        ++nv;
    }
    __device__ void begin(vec2 p) {
        first = p;
        pt(p);
        verb(3);
    }
    __device__ void end(bool close) {
        if (close) pt(first);
        verb(close ? 4 : 5);
    }
    __device__ void line_to(vec2 p) {
        pt(p);
        verb(0);
    }
    __device__ void quad_to(vec2 c, vec2 p) {
        pt(c);
        pt(p);
        verb(1);
    }
    __device__ void cubic_to(vec2 c1, vec2 c2, vec2 p) {
        pt(c1);
        pt(c2);
        pt(p);
        verb(2);
    }
};

struct PErr {
    int32_t kind, line, col;
    uint32_t ch;
};

__device__ bool parse_number(Src& S, float* v, PErr& E) {
    skip_ws(S);
    const int line = S.line, col = S.col;
    const uint32_t a = S.at;
    if (S.cur == '-') src_advance(S);
    while (is_digit(S.cur)) src_advance(S);
    if (S.cur == '.') {
        src_advance(S);
        while (is_digit(S.cur)) src_advance(S);
    }
    if (S.cur == 'e' || S.cur == 'E') {
        src_advance(S);
        if (S.cur == '-') src_advance(S);
        while (is_digit(S.cur)) src_advance(S);
    }
    const int r = parse_f32(S.s, a, S.at, v);
    if (r == NUM_OK) return true;
    E = PErr{LYG_SVG_ERR_NUMBER, line, col, 0u};
    return false;
}

__device__ bool parse_flag(Src& S, bool* f, PErr& E) {
    skip_ws(S);
    if (S.cur == '1' || S.cur == '0') {
        *f = S.cur == '1';
        src_advance(S);
        return true;
    }
    E = PErr{LYG_SVG_ERR_FLAG, S.line, S.col, S.cur};
    return false;
}

// SvgArc::to_arc (Arc::from_svg_arc, arc.rs:58-146)
__device__ ArcD svg_arc_to_arc(vec2 from, vec2 to, vec2 radii, float xrot, bool large_arc,
                               bool sweep) {
    const float PI = 3.14159265358979323846f;
    const float two_pi = 2.0f * PI;
    float rx = ffabs(radii.x), ry = ffabs(radii.y);
    const float xr = fmodf(xrot, two_pi);
    const float cos_phi = t_cos(xr), sin_phi = t_sin(xr);
    const float hd_x = (from.x - to.x) / 2.0f, hd_y = (from.y - to.y) / 2.0f;
    const float hs_x = (from.x + to.x) / 2.0f, hs_y = (from.y + to.y) / 2.0f;
    const vec2 p = mk(cos_phi * hd_x + sin_phi * hd_y, -sin_phi * hd_x + cos_phi * hd_y);
    const float rf = p.x * p.x / (rx * rx) + p.y * p.y / (ry * ry);
    if (rf > 1.0f) {
        const float scale = fsqrt(rf);
        rx *= scale;
        ry *= scale;
    }
    const float rxry = rx * ry, rxpy = rx * p.y, rypx = ry * p.x;
    const float sum_of_sq = rxpy * rxpy + rypx * rypx;
    const float sign_coe = large_arc == sweep ? -1.0f : 1.0f;
    const float coe = sign_coe * fsqrt(ffabs((rxry * rxry - sum_of_sq) / sum_of_sq));
    const float tcx = coe * rxpy / ry;
    const float tcy = -coe * rypx / rx;
    const vec2 center = mk(cos_phi * tcx - sin_phi * tcy + hs_x, sin_phi * tcx + cos_phi * tcy + hs_y);
    const vec2 start_v = mk((p.x - tcx) / rx, (p.y - tcy) / ry);
    const vec2 end_v = mk((-p.x - tcx) / rx, (-p.y - tcy) / ry);
    const float start_angle = angle_of(start_v);
    float sweep_angle = fmodf(angle_of(end_v) - start_angle, two_pi);
    if (sweep && sweep_angle < 0.0f) sweep_angle += two_pi;
    else if (!sweep && sweep_angle > 0.0f) sweep_angle -= two_pi;
    return ArcD{center, mk(rx, ry), start_angle, sweep_angle, xrot};
}

// Arguments a command reads (parser.rs:225-337): L/M/T 2, H/V 1, Q/S 4, C 6, A 7 (flags at
// 3 and 4), Z 0; -1 for a character that is no command.  Endpoint attributes come on top.
__device__ __forceinline__ int cmd_args(uint32_t c) {
    switch (c | 0x20u) {
        case 'm':
        case 'l':
        case 't':
            return 2;
        case 'h':
        case 'v':
            return 1;
        case 'q':
        case 's':
            return 4;
        case 'c':
            return 6;
        case 'a':
            return 7;
        case 'z':
            return 0;
        default:
            return -1;
    }
}

// PathParser::parse (parser.rs:154-175) and parse_path (:177-357), driven by tokens: every
// iteration of the loop reads one number or flag, so the lanes of a wave (one string each)
// spend their time in the same code whatever command each of them is in; a command is
// applied when its last argument has been read.  Relative coordinates, smooth control
// points and an arc's start use the position at the command's start, as parse_point /
// get_smooth_ctrl do (the position only changes at the command's endpoint).
template <bool EMIT>
__device__ void parse_svg(const uint8_t* s, uint32_t a, uint32_t b, int nattr, int stop_at,
                          Out<EMIT>& O, PErr& E) {
    Src S;
    src_init(S, s, a, b);
    E = PErr{LYG_SVG_OK, 0, 0, 0u};
    bool need_end = false;
    vec2 cur = mk(0.0f, 0.0f), first_pos = mk(0.0f, 0.0f);
    bool need_start = false;
    bool has_pc = false, has_pq = false;
    vec2 pc = cur, pq = cur;
    uint32_t implicit = 'M';
    uint32_t cmd = 0;
    int k = 0, nargs = 0, nums = 0;  // next argument, arguments in all, of them before attrs
    float g0 = 0, g1 = 0, g2 = 0, g3 = 0, g4 = 0, g5 = 0, g6 = 0;
    skip_ws(S);
    for (;;) {
        if (k == 0) {
            // a command boundary
            if (S.finished) break;
            uint32_t c = S.cur;
            const int cl = S.line, cc = S.col;
            if (stop_at >= 0 && (uint32_t)stop_at == c) break;
            if ((c | 0x20u) >= 'a' && (c | 0x20u) <= 'z') src_advance(S);
            else c = implicit;
            if (need_start && c != 'm' && c != 'M') {
                E = PErr{LYG_SVG_ERR_MISSING_MOVE_TO, cl, cc, c};
                break;
            }
            const int na = cmd_args(c);
            if (na < 0) {
                E = PErr{LYG_SVG_ERR_COMMAND, cl, cc, c};
                break;
            }
            cmd = c;
            if (na == 0) {
                // Z
                O.end(true);
                cur = first_pos;
                need_end = false;
                need_start = true;
                has_pc = has_pq = false;
                implicit = cmd == 'z' ? 'm' : 'M';
                skip_ws(S);
                continue;
            }
            if ((cmd | 0x20u) == 'm' && need_end) {
                O.end(false);
                need_end = false;
            }
            nums = na;
            nargs = na + nattr;
        }
        // one argument: a flag (an arc's 4th and 5th) or a number
        float v = 0.0f;
        if ((cmd | 0x20u) == 'a' && (k == 3 || k == 4)) {
            bool f;
            if (!parse_flag(S, &f, E)) break;
            v = f ? 1.0f : 0.0f;
        } else {
            if (!parse_number(S, &v, E)) break;
        }
        if (k < nums) {
            g0 = k == 0 ? v : g0;
            g1 = k == 1 ? v : g1;
            g2 = k == 2 ? v : g2;
            g3 = k == 3 ? v : g3;
            g4 = k == 4 ? v : g4;
            g5 = k == 5 ? v : g5;
            g6 = k == 6 ? v : g6;
        }
        ++k;
        if (k < nargs) continue;
        // the command's arguments are all read: apply it
        k = 0;
        const bool rel = cmd >= 'a' && cmd <= 'z';
        const vec2 o = rel ? cur : mk(0.0f, 0.0f);
        auto P = [&](float x, float y) { return rel ? mk(x + o.x, y + o.y) : mk(x, y); };
        switch (cmd | 0x20u) {
            case 'l': {
                const vec2 to = P(g0, g1);
                cur = to;
                O.line_to(to);
                break;
            }
            case 'h': {
                const vec2 to = mk(rel ? g0 + cur.x : g0, cur.y);
                cur = to;
                O.line_to(to);
                break;
            }
            case 'v': {
                const vec2 to = mk(cur.x, rel ? g0 + cur.y : g0);
                cur = to;
                O.line_to(to);
                break;
            }
            case 'q': {
                const vec2 c1 = P(g0, g1), to = P(g2, g3);
                cur = to;
                pq = c1;
                has_pq = true;
                O.quad_to(c1, to);
                break;
            }
            case 't': {
                const vec2 c1 = has_pq ? add(cur, sub(cur, pq)) : cur;
                const vec2 to = P(g0, g1);
                cur = to;
                pq = c1;
                has_pq = true;
                O.quad_to(c1, to);
                break;
            }
            case 'c': {
                const vec2 c1 = P(g0, g1), c2 = P(g2, g3), to = P(g4, g5);
                cur = to;
                pc = c2;
                has_pc = true;
                O.cubic_to(c1, c2, to);
                break;
            }
            case 's': {
                const vec2 c1 = has_pc ? add(cur, sub(cur, pc)) : cur;
                const vec2 c2 = P(g0, g1), to = P(g2, g3);
                cur = to;
                pc = c2;
                has_pc = true;
                O.cubic_to(c1, c2, to);
                break;
            }
            case 'a': {
                const vec2 from = cur;
                const vec2 to = P(g5, g6);
                cur = to;
                // Angle::degrees: f32::to_radians, x * (PI / 180)
                const float xrot = g2 * (3.14159265358979323846f / 180.0f);
                // SvgArc::is_straight_line (arc.rs:534-538)
                const float EPS = 1.1920929e-07f;
                if (ffabs(g0) <= EPS || ffabs(g1) <= EPS || veq(from, to)) {
                    O.line_to(to);
                } else {
                    const ArcD arc = svg_arc_to_arc(from, to, mk(g0, g1), xrot, g3 != 0.0f,
                                                    g4 != 0.0f);
                    arc_to_quads_each(arc, [&](int, vec2, vec2 ctrl, vec2 qto) {
                        O.quad_to(ctrl, qto);
                    });
                }
                break;
            }
            default: {  // m
                const vec2 to = P(g0, g1);
                cur = to;
                first_pos = to;
                O.begin(to);
                need_end = true;
                need_start = false;
                break;
            }
        }
        const uint32_t lc = cmd | 0x20u;
        if (lc == 'c' || lc == 's') {
            has_pq = false;
        } else if (lc == 'q' || lc == 't') {
            has_pc = false;
        } else {
            has_pc = has_pq = false;
        }
        implicit = cmd == 'm' ? 'l' : cmd == 'M' ? 'L' : cmd;
        skip_ws(S);
    }
    if (need_end) O.end(false);
    if (S.non_ascii) E = PErr{LYG_SVG_ERR_NON_ASCII, S.na_line, S.na_col, 0u};
}

// ---- a wave per string ------------------------------------------------------------------
// A string the parser accepts from beginning to end, without arcs and smooth quadratics, is a
// sequence of numbers and command letters that can be found without walking it: 64
// characters at a time, ballots tell the classes apart, and a character starts a number by
// itself, the one before it and the last one before it that is no digit.  Lanes then convert
// a number each, and a lane applies one command (or one repetition of it) each; only the
// current point goes from lane to lane, as relative commands add to it in order.  Whatever
// does not fit (errors, non-ASCII text, arcs, digits or exponents beyond the one-operation
// conversion, letters that start no command) is noticed, and the string is left to the serial
// parser below, which reports errors where they are.  That a lane's numbers are the ones the
// serial parser reads: they do not overlap, and their lengths add up to all the characters of
// numbers, so what lies between two of them is separators and command letters.
//
// Bound by VALU issue and the latency of a wave's ~90 instructions per 64 characters.  4,096
// strings of 8-64 segments (1.1 KB on average): 2,368 us with a lane per string, the text read
// byte by byte (now only for the strings left over); 72 us so.
constexpr uint32_t SVG_CHARS = 1024;  // characters looked at together
constexpr uint32_t SVG_AHEAD = 64;    // and beyond, for a number that ends there
constexpr int SVG_WAVES = 4;
// Up to here a string that its wave leaves is parsed by a lane of that wave, one launch less;
// beyond, many of them fill lanes better in a launch of their own.  us a call of 1 / 64 / 1,024
// / 4,096 strings with an arc: 329 375 546 1,127 by their waves, 369 384 560 1,050 in a launch.
constexpr uint32_t SVG_FEW = 1024;
constexpr uint32_t SVG_LEFT = 0xffffffffu;  // verbs of a string left to the serial parser

struct SvgText {
    uint8_t text[SVG_CHARS + SVG_AHEAD];
    uint16_t start[SVG_CHARS + WAVE];  // where the numbers start
};

// The number at t[p], read as the serial parser would; its end in *end.  False when it is not
// one, or not one that a double operation converts.
__device__ __forceinline__ bool wave_number(const uint8_t* t, uint32_t p, uint32_t* end, float* out) {
    const uint32_t lim = SVG_CHARS + SVG_AHEAD - 1;  // t[lim] is never part of a number read here
    uint32_t ch = t[p];
    const bool neg = ch == '-';
    if (neg) ch = t[++p];
    uint64_t w = 0;
    int kept = 0, mant = 0, shift = 0;
    bool frac = false;
    for (;;) {
        if (is_digit(ch)) {
            const uint32_t d = ch - '0';
            ++mant;
            kept += (kept != 0) | (d != 0);
            w = w * 10 + d;
            shift -= frac;
        } else if (ch == '.' && !frac) {
            frac = true;
        } else {
            break;
        }
        if (p >= lim) return false;
        ch = t[++p];
    }
    int ex = 0;
    if (ch == 'e' || ch == 'E') {
        if (p >= lim) return false;
        ch = t[++p];
        const bool eneg = ch == '-';
        if (eneg && p < lim) ch = t[++p];
        int ed = 0;
        while (is_digit(ch) && p < lim) {
            ex = ex < 100000 ? ex * 10 + (int)(ch - '0') : ex;
            ++ed;
            ch = t[++p];
        }
        if (ed == 0) return false;
        if (eneg) ex = -ex;
    }
    *end = p;
    if (mant == 0 || kept > 19 || p >= lim) return false;
    const int e = ex + shift;
    uint32_t bits;
    if (w == 0 || e + kept <= -46) bits = 0;
    else if (e + kept > 39) bits = 0x7f800000u;
    else if (!fast_round(w, e, &bits)) return false;
    *out = __uint_as_float(bits | (neg ? 0x80000000u : 0u));
    return true;
}

// Parses the string if it can; false leaves it to the serial parser.  vals, cmds: room for as
// many numbers and command words as the string has characters.
__device__ bool wave_svg(const uint8_t* s, uint32_t len, SvgText& T, float* vals, uint32_t* cmds,
                         Out<true>& O) {
    const int l = lane_id();
    if (len >= 1u << 24) return false;  // a command word holds its first number in 24 bits
    uint32_t n_num = 0, n_cmd = 0, in_numbers = 0, covered = 0, prev_end = 0;
    uint32_t last_c = ' ';
    // the last character that is no digit: 0 closes a number before a '.', 1 a sign that starts
    // one, 2 a separator or command
    uint32_t last_kind = 2;
    for (uint32_t base = 0; base < len; base += SVG_CHARS) {
        wave_sync();
        const uint32_t here = len - base < SVG_CHARS ? len - base : SVG_CHARS;
        uint32_t c[SVG_CHARS / WAVE + 1];
#pragma unroll
        for (uint32_t r = 0; r <= SVG_CHARS / WAVE; ++r) {
            const uint32_t i = base + r * WAVE + (uint32_t)l;
            c[r] = i < len ? (uint32_t)s[i] : 0u;
        }
#pragma unroll
        for (uint32_t r = 0; r <= SVG_CHARS / WAVE; ++r) T.text[r * WAVE + l] = (uint8_t)c[r];
        wave_sync();
        uint32_t n_here = 0;
        for (uint32_t r = 0; r * WAVE < here; ++r) {
            uint32_t ch = T.text[r * WAVE + l];
            if (r * WAVE + (uint32_t)l >= here) ch = ' ';
            const uint32_t lower = ch | 0x20u;
            const bool digit = is_digit(ch), dot = ch == '.', minus = ch == '-';
            const uint32_t before = from_lane_before(ch, last_c);
            const bool expo = lower == 'e' && (is_digit(before) || before == '.');
            const bool sep = is_ws(ch) || ch == ',';
            const bool cmd = lower == 'm' || lower == 'l' || lower == 'h' || lower == 'v' ||
                             lower == 'q' || lower == 's' || lower == 'c' || lower == 'z';
            if (ballot(!(digit || dot || minus || expo || sep || cmd)) != 0) return false;
            const uint64_t dm = ballot(digit), xm = ballot(expo);
            const bool exp_sign = minus && (before | 0x20u) == 'e';
            const uint64_t closing = ballot(dot || exp_sign) | xm;
            const uint64_t sign = ballot(minus && !exp_sign);
            const uint64_t below = ~dm & mask_lt(l);
            uint32_t kind = last_kind;
            if (below) {
                const int q = highest_bit(below);
                kind = (closing >> q & 1u) ? 0u : (sign >> q & 1u) ? 1u : 2u;
            }
            const bool after_sep = is_ws(before) || before == ',' ||
                                   ((before | 0x20u) >= 'a' && (before | 0x20u) <= 'z' &&
                                    (before | 0x20u) != 'e');
            const bool starts = (digit && after_sep) || (minus && !exp_sign) ||
                                (dot && (kind == 0u || (kind == 2u && !is_digit(before))));
            const uint64_t sm = ballot(starts), cm = ballot(cmd);
            const uint32_t nb = (uint32_t)__builtin_popcountll(sm & mask_lt(l));
            if (starts) T.start[n_here + nb] = (uint16_t)(r * WAVE + l);
            if (cmd)
                cmds[n_cmd + (uint32_t)__builtin_popcountll(cm & mask_lt(l))] =
                    ch << 24 | (n_num + n_here + nb);
            in_numbers += (uint32_t)__builtin_popcountll(dm | closing | sign);
            n_here += (uint32_t)__builtin_popcountll(sm);
            n_cmd += (uint32_t)__builtin_popcountll(cm);
            last_c = readlane_u(ch, WAVE - 1);
            const uint64_t other = ~dm;
            if (other) {
                const int q = highest_bit(other);
                last_kind = (closing >> q & 1u) ? 0u : (sign >> q & 1u) ? 1u : 2u;
            }
        }
        wave_sync();
        for (uint32_t k0 = 0; k0 < n_here; k0 += WAVE) {
            const uint32_t k = k0 + (uint32_t)l;
            bool bad = false;
            uint32_t n = 0, end = 0;
            if (k < n_here) {
                const uint32_t p = T.start[k];
                float v = 0.0f;
                end = p;
                bad = !wave_number(T.text, p, &end, &v);
                vals[n_num + k] = v;
                n = end - p;
                bad |= k + 1 < n_here && end > T.start[k + 1];
                bad |= k == 0 && base + p < prev_end;
            }
            if (ballot(bad) != 0) return false;
            covered += readlane_u(incl_scan(n), WAVE - 1);
            const uint32_t lastk = n_here - 1 - k0;
            if (lastk < (uint32_t)WAVE) prev_end = base + readlane_u(end, (int)lastk);
        }
        n_num += n_here;
    }
    if (covered != in_numbers) return false;
    if (n_cmd == 0) return n_num == 0;
    wave_sync();
    vec2 cur = mk(0.0f, 0.0f), first = cur, pc = cur;
    uint32_t has_pc = 0, last_cmd = 0;
    for (uint32_t g = 0; g < n_cmd; g += WAVE) {
        // a lane per command: its repetitions
        const uint32_t m = g + (uint32_t)l;
        const uint32_t word = m < n_cmd ? cmds[m] : 0u;
        const uint32_t letter = word >> 24, at = word & 0xffffffu;
        const uint32_t upto = m + 1 < n_cmd ? cmds[m + 1] & 0xffffffu : n_num;
        const uint32_t cnt = upto - at, lc = letter | 0x20u;
        const uint32_t args = lc == 'c' ? 6u : lc == 'q' || lc == 's' ? 4u
                            : lc == 'm' || lc == 'l' ? 2u : lc == 'z' ? 0u : 1u;
        uint32_t reps = 0;
        bool bad = false;
        const uint32_t before = from_lane_before(letter, last_cmd);
        if (m < n_cmd) {
            reps = args == 6u ? cnt / 6u : args == 4u ? cnt / 4u : args == 2u ? cnt / 2u : cnt;
            bad = reps * args != cnt || reps == 0u;
            if (args == 0u) {
                bad = cnt != 0u;
                reps = 1u;
            }
            // the first command, and the one after a Close, begin a sub-path; no numbers
            // come before the first
            if (m == 0) bad |= lc != 'm' || at != 0u;
            else bad |= (before | 0x20u) == 'z' && lc != 'm';
        }
        if (ballot(bad) != 0) return false;
        const uint32_t incl = incl_scan(reps), excl = incl - reps;
        const uint32_t total = readlane_u(incl, WAVE - 1);
        const uint32_t n_lanes = n_cmd - g < (uint32_t)WAVE ? n_cmd - g : (uint32_t)WAVE;
        for (uint32_t s0 = 0; s0 < total; s0 += WAVE) {
            // a lane per repetition: the last command whose first one is not past it
            const uint32_t n = total - s0 < (uint32_t)WAVE ? total - s0 : (uint32_t)WAVE;
            const uint32_t rep = s0 + (uint32_t)l;
            uint32_t j = 0;
#pragma unroll
            for (uint32_t step = 32; step; step >>= 1) {
                const uint32_t e = shfl_u(excl, (int)(j + step < 63u ? j + step : 63u));
                if (j + step < n_lanes && e <= rep) j += step;
            }
            const uint32_t L0 = shfl_u(letter, (int)j), nth = rep - shfl_u(excl, (int)j);
            const uint32_t na = shfl_u(args, (int)j);
            const uint32_t arg0 = shfl_u(at, (int)j) + nth * na;
            const uint32_t bl = shfl_u(before, (int)j);
            const bool on = (uint32_t)l < n;
            uint32_t op = L0 | 0x20u;
            const bool rel = L0 >= 'a';
            const bool move = op == 'm' && nth == 0u;
            if (op == 'm' && nth != 0u) op = 'l';
            float a[6];
#pragma unroll
            for (uint32_t q = 0; q < 6; ++q) a[q] = on && q < na ? vals[arg0 + q] : 0.0f;
            // the current point, lane to lane: set, moved, kept or back at the first point
            const vec2 v = op == 'c' ? mk(a[4], a[5])
                         : op == 'q' || op == 's' ? mk(a[2], a[3])
                         : op == 'v' ? mk(0.0f, a[0]) : mk(a[0], a[1]);
            vec2 end = v, fst = v;
            for (uint32_t q = 0; q < n; ++q) {
                const vec2 p = from_lane_before(end, cur), f = from_lane_before(fst, first);
                end.x = op == 'z' ? f.x : op == 'v' ? p.x : rel ? v.x + p.x : v.x;
                end.y = op == 'z' ? f.y : op == 'h' ? p.y : rel ? v.y + p.y : v.y;
                fst = move ? end : f;
            }
            const vec2 from = from_lane_before(end, cur);
            auto P = [&](float x, float y) { return rel ? mk(x + from.x, y + from.y) : mk(x, y); };
            const vec2 p0 = P(a[0], a[1]), p1 = P(a[2], a[3]);
            const vec2 c2 = op == 'c' ? p1 : p0;  // of a cubic
            const bool is_c = op == 'c' || op == 's';
            const vec2 pcb = from_lane_before(c2, pc);
            const bool hpc = from_lane_before(is_c ? 1u : 0u, has_pc) != 0u;
            const vec2 smooth = hpc ? add(from, sub(from, pcb)) : from;
            const bool close_before = move && (bl | 0x20u) != 'z' && bl != 0u;
            const uint32_t nv = !on ? 0u : close_before ? 2u : 1u;
            const uint32_t np = !on ? 0u : is_c ? 3u : op == 'q' ? 2u : 1u;
            const uint32_t vi = incl_scan(nv), pi = incl_scan(np);
            uint32_t ov = O.nv + vi - nv, op_ = O.np + pi - np;
            auto verb = [&](uint32_t x) {
                if (ov < O.cap_v) O.verbs[ov] = (uint8_t)x;
                ++ov;
            };
            auto point = [&](vec2 x) {
                if (op_ < O.cap_p) O.points[op_] = make_float2(x.x, x.y);
                ++op_;
            };
            if (on) {
                if (close_before) verb(5);
                verb(move ? 3u : is_c ? 2u : op == 'q' ? 1u : op == 'z' ? 4u : 0u);
                if (is_c) point(op == 'c' ? p0 : smooth);
                if (is_c) point(c2);
                if (op == 'q') point(p0);
                point(end);
            }
            O.nv += readlane_u(vi, WAVE - 1);
            O.np += readlane_u(pi, WAVE - 1);
            const int last = (int)n - 1;
            cur = readlane_v(end, last);
            first = readlane_v(fst, last);
            pc = readlane_v(c2, last);
            has_pc = readlane_u(is_c ? 1u : 0u, last);
        }
        last_cmd = readlane_u(letter, (int)n_lanes - 1);
    }
    if ((last_cmd | 0x20u) != 'z') {
        if (l == 0 && O.nv < O.cap_v) O.verbs[O.nv] = 5;
        ++O.nv;
    }
    return true;
}

}  // namespace

// Parses string i into its staging room: verbs at text_off[i] + 2 i (room: its bytes + 2),
// points at 2 text_off[i] + 2 i (room: twice its bytes + 2).  Every command consumes at
// least one character and makes at most one verb and two points per character (an arc's
// eight quadratics need eleven), plus the End of the last sub-path; a string whose output
// would not fit anyway raises the overflow counter instead of writing past its room.
__device__ __forceinline__ void serial_string(const SvgLaunch& L, uint32_t i) {
    const uint32_t a = L.text_off[i], b = L.text_off[i + 1];
    PErr E;
    Out<true> O{L.verbs + a + 2ull * i, reinterpret_cast<float2*>(L.points) + 2ull * a + 2ull * i,
                0, 0, mk(0.0f, 0.0f), b - a + 2, 2 * (b - a) + 2};
    parse_svg<true>(L.text, a, b, L.num_attributes, L.stop_at, O, E);
    L.counts_v[i] = O.nv;
    L.counts_p[i] = O.np;
    if (O.nv > O.cap_v || O.np > O.cap_p) atomicAdd(L.n_errors + 1, 1u);
    if (L.errors) {
        int32_t* e = L.errors + 4ull * i;
        e[0] = E.kind;
        e[1] = E.line;
        e[2] = E.col;
        e[3] = (int32_t)E.ch;
    }
    if (E.kind != LYG_SVG_OK) atomicAdd(L.n_errors, 1u);
}

// A wave per string; the staging rooms as serial_string's.  The upper half of a string's
// points room (twice as many as its characters; a point takes at least one) holds its numbers
// and command words meanwhile.  SERIAL: a lane of the wave goes through a string that the wave
// leaves, else svg_parse_kernel does.
template <bool SERIAL>
__global__ void __launch_bounds__(WAVE* SVG_WAVES) svg_wave_kernel(SvgLaunch L) {
    __shared__ SvgText texts[SVG_WAVES];
    const uint32_t w = readlane_u(threadIdx.x / WAVE, 0);
    const uint32_t i = blockIdx.x * SVG_WAVES + w;
    if (i >= L.n) return;
    const uint32_t a = L.text_off[i], len = L.text_off[i + 1] - a;
    float2* pts = reinterpret_cast<float2*>(L.points) + 2ull * a + 2ull * i;
    float* vals = reinterpret_cast<float*>(pts + len + 2u);
    Out<true> O{L.verbs + a + 2ull * i, pts, 0, 0, mk(0.0f, 0.0f), len + 2, 2 * len + 2};
    const bool done = wave_svg(L.text + a, len, texts[w], vals,
                               reinterpret_cast<uint32_t*>(vals) + len, O);
    // what the wave wrote of a string it leaves comes before what the lane writes there
    if (SERIAL && !done) __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    if (lane_id() != 0) return;
    if (!done) {
        if (SERIAL) serial_string(L, i);
        else L.counts_v[i] = SVG_LEFT;
        return;
    }
    L.counts_v[i] = O.nv;
    L.counts_p[i] = O.np;
    if (O.nv > O.cap_v || O.np > len + 2u) atomicAdd(L.n_errors + 1, 1u);
    if (L.errors)
        for (int k = 0; k < 4; ++k) L.errors[4ull * i + k] = 0;
}

// The serial parser, a lane per string; of the strings left by the wave parser, the block's
// first lanes take those among its 256 (a list of them all through one counter cost 45 us when
// all of 4,096 strings were left).
__global__ void __launch_bounds__(256) svg_parse_kernel(SvgLaunch L) {
    __shared__ uint32_t left[256], n_left;
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (L.by_wave) {
        if (threadIdx.x == 0) n_left = 0;
        __syncthreads();
        if (i < L.n && L.counts_v[i] == SVG_LEFT) left[atomicAdd(&n_left, 1u)] = i;
        __syncthreads();
        if (threadIdx.x >= n_left) return;
        i = left[threadIdx.x];
    } else if (i >= L.n) {
        return;
    }
    serial_string(L, i);
}

// Copies every string's verbs and points from its staging room to its place in the batch:
// one block per string.
__global__ void __launch_bounds__(256) svg_compact_kernel(SvgLaunch L, uint8_t* verbs,
                                                          float* points) {
    for (uint32_t i = blockIdx.x; i < L.n; i += gridDim.x) {
        const uint32_t a = L.text_off[i];
        const uint8_t* sv = L.verbs + a + 2ull * i;
        const float2* sp = reinterpret_cast<const float2*>(L.points) + 2ull * a + 2ull * i;
        const uint32_t ov = L.off_v[i], nv = L.off_v[i + 1] - ov;
        const uint32_t op = L.off_p[i], np = L.off_p[i + 1] - op;
        for (uint32_t k = threadIdx.x; k < nv; k += blockDim.x) verbs[ov + k] = sv[k];
        float2* dp = reinterpret_cast<float2*>(points) + op;
        for (uint32_t k = threadIdx.x; k < np; k += blockDim.x) dp[k] = sp[k];
    }
}

}  // namespace lyg

extern "C" {

hipError_t lyg_launch_svg_parse(const lyg::SvgLaunch* L, hipStream_t s) {
    using namespace lyg;
    if (L->n == 0) return hipSuccess;
    if (L->by_wave) {
        const dim3 grid((L->n - 1) / SVG_WAVES + 1), block(WAVE * SVG_WAVES);
        if (L->n <= SVG_FEW) {
            hipLaunchKernelGGL(svg_wave_kernel<true>, grid, block, 0, s, *L);
            return hipGetLastError();
        }
        hipLaunchKernelGGL(svg_wave_kernel<false>, grid, block, 0, s, *L);
    }
    hipLaunchKernelGGL(svg_parse_kernel, dim3((L->n + 255) / 256), dim3(256), 0, s, *L);
    return hipGetLastError();
}

hipError_t lyg_launch_svg_compact(const lyg::SvgLaunch* L, uint8_t* verbs, float* points,
                                  hipStream_t s) {
    if (L->n == 0) return hipSuccess;
    const uint32_t blocks = L->n < 65536u ? L->n : 65536u;
    hipLaunchKernelGGL(lyg::svg_compact_kernel, dim3(blocks), dim3(256), 0, s, *L, verbs, points);
    return hipGetLastError();
}

}  // extern "C"
