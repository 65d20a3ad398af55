// Checks the word reads of image tiles (word_place, lbsp_form in bgs_common.hpp) on the host: every read lies
// inside the buffer and yields the buffer's bytes, zeros beside them. Prints "ok" and the number of reads.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../../litiv_amd/csrc/bgs_common.hpp"

using namespace lvbgs;

static long reads = 0;

#define CHECK(c, ...)                       \
    do {                                    \
        if (!(c)) {                         \
            std::printf(__VA_ARGS__);       \
            std::printf(" (%s)\n", #c);     \
            std::exit(1);                   \
        }                                   \
    } while (0)

// a read at `off` of a buffer of these bytes
template <typename I>
static void read_word(const std::vector<unsigned char>& buf, I off) {
    const I total = (I)buf.size();
    const I at = word_place(off, total), beyond = off - at;
    CHECK(at >= 0 && at + 4 <= total, "total %ld off %ld reads from %ld", (long)total, (long)off, (long)at);
    uint32_t w = 0, want = 0;
    for (int k = 0; k < 4; ++k) w |= (uint32_t)buf[(size_t)(at + k)] << (8 * k);
    w = beyond < 0 || beyond > 3 ? 0u : w >> (8 * (int)beyond);
    for (int k = 0; k < 4; ++k)
        if (off >= 0 && off + k < total) want |= (uint32_t)buf[(size_t)(off + k)] << (8 * k);
    CHECK(w == want, "total %ld off %ld: %08x, not %08x", (long)total, (long)off, w, want);
    ++reads;
}

int main() {
    // small images: the offsets that tiles of 64x4 pixels with a halo of 2 read
    for (int H = 1; H <= 9; ++H)
        for (int W = 1; W <= 70; W = W < 9 ? W + 1 : W + 13)
            for (int C = 1; C <= 3; C += 2) {
                const LbspForm form = lbsp_form(W, H, C);
                CHECK((form == kLbspEmpty) == (W < 5 || H < 5), "%dx%dx%d", W, H, C);
                if (form == kLbspEmpty) continue;
                CHECK(form == kLbsp32, "%dx%dx%d", W, H, C);
                std::vector<unsigned char> buf((size_t)W * H * C);
                for (size_t i = 0; i < buf.size(); ++i) buf[i] = (unsigned char)(i * 37 + 11);
                for (int gy = 0; gy < H; ++gy)
                    for (int x0 = 0; x0 < W; x0 += 64)
                        for (int k = 0; k < 72; ++k) {
                            const int off = C == 3 ? (gy * W + x0 + k - 2) * 3 : gy * W + x0 - 4 + k;
                            read_word<int>(buf, off);
                            read_word<int64_t>(buf, off);
                        }
            }
    // large images: the furthest offset of the 32-bit form fits, and the 64-bit one starts where it need not
    const int sizes[][3] = {{46340, 46336, 1}, {46341, 46341, 1}, {26754, 26754, 3}, {26755, 26755, 3}, {5, 429496678, 1},
                            {5, 429496679, 1}, {715827797, 5, 3}, {143165500, 5, 3}};
    for (const auto& s : sizes) {
        const int64_t W = s[0], H = s[1], C = s[2], total = W * H * C;
        const LbspForm form = lbsp_form(s[0], s[1], s[2]);
        const int64_t far = ((H - 1) * W + (W + 63) / 64 * 64 + 4) * C + 4;
        CHECK(form == kLbsp64 || far <= 0x7FFFFFFFll, "%dx%dx%d", s[0], s[1], s[2]);
        CHECK(form == kLbsp32 || total > 0x7FFFFFFFll - 256, "%dx%dx%d", s[0], s[1], s[2]);
        for (int64_t d = -300; d <= 300; ++d) {
            const int64_t at = word_place<int64_t>(total + d, total);
            CHECK(at >= 0 && at + 4 <= total, "%dx%dx%d", s[0], s[1], s[2]);
        }
    }
    std::printf("ok %ld\n", reads);
}
