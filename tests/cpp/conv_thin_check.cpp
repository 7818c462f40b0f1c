// Host-side checks of helix_conv_thin.h.
//   conv_thin_check windows: the loads of every unit of four pixels lie inside x, and the dwords they leave after being
//     moved hold the unit's halves, for every x of 8 to 40 pixels and every pixel a unit can start at;
//   conv_thin_check plans < layers: one line per layer read (batch IC H W OC kH kW stride pad), 1 if the kernel takes it.
#include <stdio.h>
#include <string.h>

#include "helix_conv_thin.h"

static int windows() {
    long bad = 0;
    for (int pixels = 8; pixels <= 40; pixels++) {
        const int bytes = pixels * 6;
        unsigned char x[256];
        for (int i = 0; i < bytes; i++) x[i] = (unsigned char)(i * 7 + 1);
        for (int pixel = 0; pixel < pixels; pixel++) {
            const int at = pixel * 6;
            const helix_conv_thin::Window n = helix_conv_thin::window_of(at, bytes);
            if (n.from < 0 || n.from % 4 || n.from + 28 > bytes || n.behind < 0 || n.behind > 6) {
                bad++;
                continue;
            }
            unsigned w[7];
            memcpy(w, x + n.from, 28);
            for (int b = 0; b < n.behind; b++) {
                for (int e = 0; e < 6; e++) w[e] = w[e + 1];
                w[6] = (unsigned)x[bytes - 2] | (unsigned)x[bytes - 1] << 8;
            }
            const int held = bytes - at < 24 ? bytes - at : 24;      // what of the unit lies in x
            bad += memcmp((unsigned char*)w + (at & 2), x + at, held) != 0;
        }
    }
    printf("mismatches %ld\n", bad);
    return bad != 0;
}

int main(int argc, char** argv) {
    if (argc == 2 && !strcmp(argv[1], "windows")) return windows();
    int l[9];
    while (scanf("%d %d %d %d %d %d %d %d %d", l, l + 1, l + 2, l + 3, l + 4, l + 5, l + 6, l + 7, l + 8) == 9) {
        helix_conv_thin::Plan plan;
        printf("%d\n", (int)helix_conv_thin::make_plan(plan, l[0], l[2], l[3], l[1], l[4], l[5], l[6], l[7], l[8]));
    }
    return 0;
}
