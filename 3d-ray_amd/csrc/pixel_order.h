// pixel_order.h — order of a window's pixels and of a launch's workgroups.
// Plain C++ besides RT_HD, which the including file defines.
#pragma once
#include <stdint.h>

namespace rt {

// Pixel order of a window's samples: strips of 8 rows, column by column
// inside a strip (64 consecutive pixels are an 8 x 8 tile); the last strip
// takes the rows that are left, an image of fewer rows is one strip (so that
// a strip's pixels, at most the image's, fit an int).
constexpr int kStripRows = 8;
RT_HD int pixel_of_rank(int q, int W, int npix) {
    const int H = npix / W, rows = H < kStripRows ? H : kStripRows;
    const int strip = q / (rows * W), y0 = strip * rows;
    const int r = q - y0 * W, left = H - y0, h = left < rows ? left : rows;
    const int x = r / h;
    return (y0 + r - x * h) * W + x;
}

// XCD-aware block order: gfx950 dispatches consecutive workgroups round-robin
// over its 8 XCDs; renumber so each XCD walks runs of consecutive blocks
// (neighbouring rays share BVH nodes in that XCD's L2) while the eight stay
// side by side in the pool, so sky and object parts of the image load them
// evenly (one eighth of the pool per XCD ran the 1080p frame in 349 instead of
// 298 ms).  Runs of `longest` blocks (2048 slots), in small pools of a 64th of
// an XCD's share, but a quarter of `longest` at least, and the XCDs change
// places from one eight of runs to the next: in a fixed order an image whose
// strips are 4 or 8 runs long gives an XCD the same columns of every strip
// (341x206 x 3 Cornell box, sky on both sides: 1.77 ms, 1.53 with an eighth of
// the pool each, 1.54 here).
constexpr uint32_t kXcdSlots = 2048;
RT_HD uint32_t xcd_remap(uint32_t b, uint32_t nb, uint32_t longest) {
    const uint32_t share = nb / 512u, least = (longest + 3u) / 4u;
    const uint32_t run = share < least ? least : share < longest ? share : longest;
    const uint32_t whole = nb / (8u * run) * (8u * run);
    if (b >= whole) return b;   // the last, partial round keeps its order
    const uint32_t i = b / 8u, eight = i / run;
    return (eight * 8u + (b + eight) % 8u) * run + i % run;
}

}  // namespace rt
