// pixel_order.h — order of a window's pixels.  Plain C++ besides RT_HD, which
// the including file defines.
#pragma once

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

}  // namespace rt
