// host_rules.h -- host-side rules that need neither HIP nor a device.
#pragma once

#include <stddef.h>

#include <initializer_list>

namespace skm {

// A workspace of several buffers: grab(&p, bytes) each (0 or an error code),
// or none of them -- after a failure the ones already there are dropped and
// null, so that a later call sees no half of a workspace.
struct Buffer {
    void** p;
    size_t bytes;
};
template <typename Grab, typename Drop>
int grab_all(std::initializer_list<Buffer> list, Grab grab, Drop drop)
{
    for (const Buffer* b = list.begin(); b != list.end(); ++b) {
        const int rc = grab(b->p, b->bytes);
        if (rc == 0) continue;
        *b->p = nullptr;
        while (b != list.begin()) {
            --b;
            drop(*b->p);
            *b->p = nullptr;
        }
        return rc;
    }
    return 0;
}

// Rows that one launch of k_screen_wide takes: their two largest values of
// every 128 centres, 16 bytes a row and 256 centres, stay under kWidePartBytes
// (a launch then has at most 65,536 blocks, 256 rounds of the CUs: what a
// launch costs and the round that it leaves partly idle are lost in them).
// All rows at once would take 8 times X for 65,536 centres of 132 floats, and
// from 8.4M blocks of 512 threads a launch is refused.
constexpr size_t kWidePartBytes = size_t(256) << 20;
inline long wide_rows(long n, int k)
{
    const long ncg = (k + 255) / 256;
    const long rows = (long)(kWidePartBytes / size_t(16 * ncg)) / 2048 * 2048;  // 256 for each of 8 XCDs
    return n < rows ? n : rows < 2048 ? 2048 : rows;
}
inline size_t wide_part_floats(long rows, int k) { return size_t(rows) * ((size_t(k) + 255) / 256) * 4; }
// k_screen_wide's blocks for `rows` rows: whole turns of the XCDs.
inline long wide_blocks(long rows, int k) { return ((rows + 255) / 256 + 7) / 8 * 8 * ((k + 255) / 256); }

// Where a run's steps begin behind the screen (screen_lost then tells whether
// they stay there).  k_assign3 alone takes its 256-row blocks in rounds
// of 256 (one a CU), each round proportional to the padded centres times
// features (0.64 us per 1,000).  Rows of at most 128 floats: what is left
// costs about one round again (nearly every block has a row) and the second
// launch and its image 20 us, so it is the rounds after the first that are
// saved.  Timed, a step without / with the screen: 64 floats, k = 1,024:
// 60,000 rows 92 / 107 us, 120,000 134 / 111, 1,000,000 693 / 311; 128
// floats, k = 256: 120,000 91 / 89, 250,000 144 / 114, 1,000,000 442 / 280.
// Longer rows: the rest goes by units of 256 rows x 256 centres and costs
// little, but there are two more launches.  768 floats, k = 1,500: 8,000 rows
// 610 / 126; 300 floats: k = 600, 8,000 rows 161 / 87; k = 200, 130,000 rows
// 158 / 142, 400,000 444 / 337; k = 512, 64,000 rows 150 / 124, 130,000 251 /
// 175.  What is left depends on the data, not on the shape.  64,000 rows of 400 to
// 768 floats, k = 400, at the second step: 2 to 3% of overlapping blobs from
// their means as centres, 95% of the same from rows of X, half of blobs a
// little further apart, from rows too.  With at most two groups of 256 centres
// and more row blocks than one round of their units (32,768 rows) the two steps
// looked at cost most: 64,000 x 768, k = 400, three steps of the 95% kind 1,165 us
// without the screen and 1,527 with, ten steps from the means 1,435 and 1,003;
// 130,000 x 640 1,934 and 2,586, 2,926 and 1,709; 33,000 x 640, k = 300 (one
// round) 926 and 908, 1,628 and 1,103.  Rows of more than 512 floats, where those
// two steps are longest, begin without the screen there; of 64,000 x 512 the same
// runs take 861 and 1,133, 1,545 and 1,055, and begin with it.
inline bool screen_pays(long n, int ld, int k)
{
    if (n >= (1L << 31) || k <= 128) return false;
    if (ld > 512 && k <= 512 && n > 32768) return false;
    const double round = (double)((k + 255) / 256 * 256) * ((ld + 31) / 32 * 32);
    const double rounds = (double)((n + 65535) / 65536);
    return ld <= 128 ? (rounds - 1) * round >= 60e3 : rounds * round >= 230e3;
}

// The E-step's time in us on 256 CUs, fitted to timings of 35 shapes (60,000 to
// 4M rows of 32 to 128 floats, 4,000 to 1M of 200 to 1,000, 200 to 4,096
// centres; within 15%, but for rows of 32 floats, and for fewer row blocks than
// CUs, where plain is up to 20% less).  plain: k_assign3, 14 us and 4.45 to 4.7
// for 32 features of 256 centres of a round of 256-row blocks.  screen: k_screen
// or k_screen_wide (4 us a block and 2.25 for 64 features, or X's bytes, of which
// rows off the cache lines cost more) with the centres' images and the empty
// launches behind it.  rest: the six products of the rows left; `passes` is
// k_assign3_list's busiest block's, which k_assign3_units (long rows) has not:
// its units of 256 centres, or of 64 where those would leave half the CUs idle,
// go round the CUs.
inline double plain_us(long n, int ld, int k)
{
    const long rounds = (n + 65535) / 65536, steps = (long)((k + 255) / 256) * ((ld + 31) / 32);
    return 14.0 + (ld <= 128 ? 4.7 : 4.45) * (double)(rounds * steps);
}
inline double screen_us(long n, int ld, int k)
{
    const double bytes = 4.0 * (double)n * ld;
    if (ld <= 128) {
        const double values = (double)n * ((k + 127) / 128 * 128), mac = values * ((ld + 31) / 32 * 32);
        const double t = mac * 1.95e-9 > values * 8.8e-8 ? mac * 1.95e-9 : values * 8.8e-8;
        return 26.0 + (t > bytes / 5.3e6 ? t : bytes / 5.3e6);
    }
    const double t = (4.0 + 2.25 * ((ld + 63) / 64)) * (double)((wide_blocks(n, k) + 255) / 256);
    const double m = bytes * (ld % 32 != 0 ? 1.4 : 1.0) / 5e6;
    return 35.0 + (t > m ? t : m);
}
inline double rest_us(long n, int ld, int k, long left, long passes)
{
    if (ld <= 128) return (double)passes * (plain_us(n, ld, k) - 14.0) / (double)((n + 65535) / 65536);
    const long units = (left + 255) / 256 * ((k + 255) / 256);
    const double unit = 4.95 * ((ld + 31) / 32);
    return units * 2 <= 256 ? 0.33 * unit * (double)((units * 4 + 255) / 256) : unit * (double)((units + 255) / 256);
}
// Whether a step that left these rows took longer than without the screen.
// Timed with the rows left spread evenly, without / with the screen, at shares
// before the line and past it: 1M x 128, k = 256 (9 passes of 16) 338 / 285 and
// 336 / 319; 250,000 x 128, k = 256 (1 of 4) 96 / 65 and 95 / 70; 1M x 64, k =
// 1,024 (11 of 16) 650 / 543 and 640 / 601; 400,000 x 300, k = 200 (a half) 327 /
// 296 and 330 / 399; 64,000 x 768, k = 400 (a half) 218 / 205 and 216 / 302;
// 100,000 x 768, k = 2,048 (four fifths) 1,544 / 1,396 and 1,545 / 1,647; 500,000
// x 768, k = 4,096 (two thirds) 13,760 / 12,227 and 13,773 / 15,280.  Rows left
// in one stretch, a tenth of 1M x 128: 338 / 404.
inline bool screen_lost(long n, int ld, int k, long left, long passes)
{
    return screen_us(n, ld, k) + rest_us(n, ld, k, left, passes) > 0.98 * plain_us(n, ld, k);
}

}  // namespace skm
