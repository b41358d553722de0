// Prints the strip height and bands that a launch takes where only the strip
// width is set: "<width> <height> <plane format> <strip_cols> <pairs>" lines on
// stdin, pairs 0 for a pipeline's pair, else a batch's on 256 CUs.
#include <iostream>

#include "ss2_host.h"

using namespace vqm::ss2;

int main() {
    uint32_t w, h, format, cols, pairs;
    while (std::cin >> w >> h >> format >> cols >> pairs) {
        const auto f = static_cast<PlaneFormat>(format);
        const ScaleShape s = pairs == 0 ? ScaleShape{SinglePairStripRows(w, h, f, 0, cols), cols,
                                                     SinglePairRowParts(w, h, f, 0, cols)}
                                        : DefaultShape(w, h, f, cols, pairs, 256, false);
        std::cout << s.rows << " " << s.row_parts << "\n";
    }
}
