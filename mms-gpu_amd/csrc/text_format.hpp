// text_format.hpp -- printf's %g of a float (six significant digits, the
// exactly rounded decimal, ties to even), for the device and the host.
//
// The digits are the integer nearest to |v| 10^k, k = 5 - floor(log10 |v|).
// 10^0 .. 10^22 are doubles, so for k >= 0 the product is exact as the sum of
// two doubles, and for -22 <= k < 0 the remainder of the division is; ties
// are seen exactly.  Further out no float lies on a tie and 10^k as two
// doubles (about 106 bits) decides.  Agrees with glibc's snprintf on all 2^32
// float bit patterns.
#pragma once
#include <math.h>
#include <stdint.h>
#include <string.h>

#ifdef __HIPCC__
#define MMS_HD __host__ __device__ inline
#else
#define MMS_HD inline
#endif

namespace mms {

// 10^k as hi + lo, k = -45 .. 50
struct Pow10 { double hi, lo; };
#define MMS_POW10_FIRST (-45)
#define MMS_POW10_ROWS \
    {0x1.6d601ad376ab9p-150, 0x1.a27ac0f72f8c0p-206}, {0x1.c8b8218854567p-147, 0x1.82c65c4d3edbcp-201}, \
    {0x1.1d7314f534b61p-143, -0x1.8e44064fb8b6bp-197}, {0x1.64cfda3281e39p-140, -0x1.e3aa0fc74dc8ap-195}, \
    {0x1.be03d0bf225c7p-137, -0x1.72524ee484eb4p-194}, {0x1.16c262777579cp-133, 0x1.631191d6259dap-187}, \
    {0x1.5c72fb1552d83p-130, 0x1.bbd5f64baf050p-184}, {0x1.b38fb9daa78e4p-127, 0x1.2acb73de9ac65p-181}, \
    {0x1.1039d428a8b8fp-123, -0x1.4540d794df441p-177}, {0x1.54484932d2e72p-120, 0x1.696ef285e8eafp-174}, \
    {0x1.a95a5b7f87a0fp-117, -0x1.e1aa86c4e6d2fp-174}, {0x1.09d8792fb4c49p-113, 0x1.5a5ead789df78p-167}, \
    {0x1.4c4e977ba1f5cp-110, -0x1.4f09a7293a8aap-164}, {0x1.9f623d5a8a733p-107, -0x1.a2cc10f3892d4p-161}, \
    {0x1.039d665896880p-103, -0x1.85bf8a9835bc4p-157}, {0x1.4484bfeebc2a0p-100, -0x1.e72f6d3e432b6p-154}, \
    {0x1.95a5efea6b347p-97, 0x1.9f04b7722c09dp-151}, {0x1.fb0f6be506019p-94, 0x1.06c5e54eb70c4p-148}, \
    {0x1.3ce9a36f23c10p-90, -0x1.b788a15d9b30bp-145}, {0x1.8c240c4aecb14p-87, -0x1.12b564da80fe7p-141}, \
    {0x1.ef2d0f5da7dd9p-84, -0x1.5762be11213e0p-138}, {0x1.357c299a88ea7p-80, 0x1.a96249354b394p-134}, \
    {0x1.82db34012b251p-77, 0x1.13badb829e079p-131}, {0x1.e392010175ee6p-74, -0x1.a7566d9cba769p-128}, \
    {0x1.2e3b40a0e9b4fp-70, 0x1.f769fb7e0b75ep-124}, {0x1.79ca10c924223p-67, 0x1.75447a5d8e536p-121}, \
    {0x1.d83c94fb6d2acp-64, 0x1.a52b31e9e3d07p-119}, {0x1.2725dd1d243acp-60, -0x1.7c628066e8ceep-114}, \
    {0x1.70ef54646d497p-57, -0x1.db7b2080a3029p-111}, {0x1.cd2b297d889bcp-54, 0x1.5b4c2ebe68799p-109}, \
    {0x1.203af9ee75616p-50, -0x1.937831647f5a0p-104}, {0x1.6849b86a12b9bp-47, 0x1.ea70909833de7p-107}, \
    {0x1.c25c268497682p-44, -0x1.ecd79a5a0df95p-99}, {0x1.19799812dea11p-40, 0x1.97f27f0f6e886p-96}, \
    {0x1.5fd7fe1796495p-37, 0x1.7f7bc7b4d28aap-91}, {0x1.b7cdfd9d7bdbbp-34, -0x1.20a5465df8d2cp-88}, \
    {0x1.12e0be826d695p-30, -0x1.34674bfabb83bp-84}, {0x1.5798ee2308c3ap-27, -0x1.03023df2d4c94p-82}, \
    {0x1.ad7f29abcaf48p-24, 0x1.5e1e99483b023p-78}, {0x1.0c6f7a0b5ed8dp-20, 0x1.b5a63f9a49c2cp-75}, \
    {0x1.4f8b588e368f1p-17, -0x1.ee78183f91e64p-71}, {0x1.a36e2eb1c432dp-14, -0x1.6a161e4f765fep-68}, \
    {0x1.0624dd2f1a9fcp-10, -0x1.89374bc6a7efap-66}, {0x1.47ae147ae147bp-7, -0x1.eb851eb851eb8p-63}, \
    {0x1.999999999999ap-4, -0x1.999999999999ap-58}, {0x1.0000000000000p+0, 0x0.0p+0}, \
    {0x1.4000000000000p+3, 0x0.0p+0}, {0x1.9000000000000p+6, 0x0.0p+0}, \
    {0x1.f400000000000p+9, 0x0.0p+0}, {0x1.3880000000000p+13, 0x0.0p+0}, \
    {0x1.86a0000000000p+16, 0x0.0p+0}, {0x1.e848000000000p+19, 0x0.0p+0}, \
    {0x1.312d000000000p+23, 0x0.0p+0}, {0x1.7d78400000000p+26, 0x0.0p+0}, \
    {0x1.dcd6500000000p+29, 0x0.0p+0}, {0x1.2a05f20000000p+33, 0x0.0p+0}, \
    {0x1.74876e8000000p+36, 0x0.0p+0}, {0x1.d1a94a2000000p+39, 0x0.0p+0}, \
    {0x1.2309ce5400000p+43, 0x0.0p+0}, {0x1.6bcc41e900000p+46, 0x0.0p+0}, \
    {0x1.c6bf526340000p+49, 0x0.0p+0}, {0x1.1c37937e08000p+53, 0x0.0p+0}, \
    {0x1.6345785d8a000p+56, 0x0.0p+0}, {0x1.bc16d674ec800p+59, 0x0.0p+0}, \
    {0x1.158e460913d00p+63, 0x0.0p+0}, {0x1.5af1d78b58c40p+66, 0x0.0p+0}, \
    {0x1.b1ae4d6e2ef50p+69, 0x0.0p+0}, {0x1.0f0cf064dd592p+73, 0x0.0p+0}, \
    {0x1.52d02c7e14af6p+76, 0x1.0000000000000p+23}, {0x1.a784379d99db4p+79, 0x1.0000000000000p+24}, \
    {0x1.08b2a2c280291p+83, -0x1.b000000000000p+29}, {0x1.4adf4b7320335p+86, -0x1.1c00000000000p+32}, \
    {0x1.9d971e4fe8402p+89, -0x1.8c00000000000p+33}, {0x1.027e72f1f1281p+93, 0x1.8440000000000p+38}, \
    {0x1.431e0fae6d721p+96, 0x1.f2a8000000000p+42}, {0x1.93e5939a08ceap+99, -0x1.215c000000000p+44}, \
    {0x1.f8def8808b024p+102, 0x1.4b26800000000p+48}, {0x1.3b8b5b5056e17p+106, -0x1.3107f00000000p+52}, \
    {0x1.8a6e32246c99cp+109, 0x1.82b6140000000p+55}, {0x1.ed09bead87c03p+112, 0x1.e363990000000p+58}, \
    {0x1.3426172c74d82p+116, 0x1.5c3c7f4000000p+61}, {0x1.812f9cf7920e3p+119, -0x1.265a307800000p+65}, \
    {0x1.e17b84357691bp+122, 0x1.900f436a00000p+68}, {0x1.2ced32a16a1b1p+126, 0x1.e826288900000p+70}, \
    {0x1.78287f49c4a1dp+129, 0x1.988becaad0000p+75}, {0x1.d6329f1c35ca5p+132, -0x1.0151182a7c000p+78}, \
    {0x1.25dfa371a19e7p+136, -0x1.069578d46c000p+79}, {0x1.6f578c4e0a061p+139, -0x1.29075ae130e00p+85}, \
    {0x1.cb2d6f618c879p+142, -0x1.cd24c665f4600p+86}, {0x1.1efc659cf7d4cp+146, -0x1.c80dbeffee2f0p+92}, \
    {0x1.66bb7f0435c9ep+149, 0x1.c5eed14016454p+95}, {0x1.c06a5ec5433c6p+152, 0x1.bb542c80deb48p+95}, \
    {0x1.18427b3b4a05cp+156, -0x1.babad90bdd33dp+101}, {0x1.5e531a0a1c873p+159, -0x1.14b4c7a76a406p+105}, \
    {0x1.b5e7e08ca3a8fp+162, 0x1.a61e066ebb2f9p+108}, {0x1.11b0ec57e649ap+166, -0x1.782d3bfacb025p+112}

// One formatted number: digits d (leading digit first in the decimal integer,
// nd of them, trailing zeros removed), exponent x of the leading digit.
struct GNum {
    uint32_t digits;  // the nd significant digits as an integer
    int8_t nd;        // 0: not a finite non-zero number, see kind
    int8_t x;
    uint8_t neg;
    uint8_t kind;     // 0 zero, 1 finite, 2 inf, 3 nan
};

MMS_HD GNum g_split(float v, const Pow10 *p10) {
    GNum g;
    uint32_t u;
    memcpy(&u, &v, 4);
    g.neg = (uint8_t)(u >> 31);
    g.digits = 0; g.nd = 0; g.x = 0;
    u &= 0x7fffffffu;
    if (u >= 0x7f800000u) { g.kind = u == 0x7f800000u ? 2 : 3; return g; }
    if (u == 0) { g.kind = 0; return g; }
    g.kind = 1;
    memcpy(&v, &u, 4);
    const double d = (double)v;
    // floor(log10 d) from the binary exponent, one too small at most
    uint64_t w;
    memcpy(&w, &d, 8);
    const int e2 = (int)(w >> 52) - 1023;
    int x = (int)floor((double)e2 * 0.30102999566398119521);
    if (d >= p10[x + 1 - MMS_POW10_FIRST].hi) x++;
    int64_t n;
    for (;;) {
        const int k = 5 - x;
        double s;
        if (k >= 0 || k < -22) {
            const Pow10 p = p10[k - MMS_POW10_FIRST];
            const double h = d * p.hi, l = fma(d, p.hi, -h) + d * p.lo, f = floor(h);
            n = (int64_t)f;
            s = ((h - f) - 0.5) + l;  // the sign of the sum of two doubles is exact
        } else {
            const double p = p10[-k - MMS_POW10_FIRST].hi;
            double f = floor(d / p), r = fma(-f, p, d);
            if (r < 0) { f -= 1; r += p; }
            else if (r >= p) { f += 1; r -= p; }
            n = (int64_t)f;
            s = r - 0.5 * p;
        }
        if (s > 0 || (s == 0 && (n & 1))) n++;
        if (n < 1000000) break;
        x++;  // rounded up to a power of ten (or x was too small): once more
    }
    g.x = (int8_t)x;
    int nd = 6;
    uint32_t q = (uint32_t)n;
    while (nd > 1 && q % 10 == 0) { q /= 10; nd--; }
    g.digits = q;
    g.nd = (int8_t)nd;
    return g;
}

MMS_HD int g_length(const GNum &g) {
    if (g.kind == 0) return 1 + g.neg;
    if (g.kind >= 2) return 3 + g.neg;
    if (g.x < -4 || g.x >= 6)  // d.ddde+xx
        return g.neg + g.nd + (g.nd > 1 ? 1 : 0) + 4;
    if (g.x < 0) return g.neg + 1 - g.x + g.nd;                    // 0.000ddd
    if (g.nd <= g.x + 1) return g.neg + g.x + 1;                   // ddd000
    return g.neg + g.nd + 1;                                       // dd.ddd
}

// writes g_length(g) characters at o
MMS_HD void g_write(const GNum &g, char *o) {
    if (g.neg) *o++ = '-';
    if (g.kind == 0) { *o = '0'; return; }
    if (g.kind >= 2) {
        const char *t = g.kind == 2 ? "inf" : "nan";
        o[0] = t[0]; o[1] = t[1]; o[2] = t[2];
        return;
    }
    uint32_t q = g.digits;
    const int nd = g.nd;
    if (g.x < -4 || g.x >= 6) {
        for (int i = nd - 1; i >= 1; i--) { o[i + 1] = (char)('0' + q % 10); q /= 10; }
        o[0] = (char)('0' + q);
        if (nd > 1) { o[1] = '.'; o += nd + 1; } else { o += 1; }
        int x = g.x;
        o[0] = 'e';
        o[1] = x < 0 ? '-' : '+';
        if (x < 0) x = -x;
        o[2] = (char)('0' + x / 10);
        o[3] = (char)('0' + x % 10);
    } else if (g.x < 0) {
        o[0] = '0'; o[1] = '.';
        o += 2;
        for (int i = -1; i > g.x; i--) *o++ = '0';
        for (int i = nd - 1; i >= 0; i--) { o[i] = (char)('0' + q % 10); q /= 10; }
    } else if (nd <= g.x + 1) {
        for (int i = g.x; i >= nd; i--) o[i] = '0';
        for (int i = nd - 1; i >= 0; i--) { o[i] = (char)('0' + q % 10); q /= 10; }
    } else {
        const int p = g.x + 1;  // digits before the point
        for (int i = nd - 1; i >= p; i--) { o[i + 1] = (char)('0' + q % 10); q /= 10; }
        o[p] = '.';
        for (int i = p - 1; i >= 0; i--) { o[i] = (char)('0' + q % 10); q /= 10; }
    }
}

}  // namespace mms
