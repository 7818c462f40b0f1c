// Host side of conv_patch.hip, one configuration of it: per layer read (batch IC H W OC kH kW stride pad) one line with the
// LDS bytes, the staged bytes and the workgroups of its plan, or "none"; exits with 1 when a block of output pixels would
// write or read beyond what the plan reserves.
#include "conv_patch.hip"

// A weight of a channel that is not there in a K chunk that is not there either: its offset is the sum of two that read zeros, in
// defined arithmetic (a signed sum would be none, and no constant), and reads zeros itself, up to the last byte of a load.
constexpr auto TWICE_OUT = OOB + OOB;
static_assert((unsigned long long)TWICE_OUT >= (unsigned long long)OOB && TWICE_OUT <= 0xffffffffu - 15, "beyond any buffer");

static int staged_row(const Params& p, int m) {
    const int t = m / p.by_OW.d, image = t / p.OH;
    return image * p.image_rows + (t - image * p.OH) * p.stride;
}

// Whether every operand that a lane reads lies inside the plan's LDS: all entries of the table, those of the K tile that is read
// ahead (and by a wave whose part of K is empty) among them, for pixels whose corners are at `first` .. `last`.
template <bool REST>
static bool operands_inside(const Params& p, int first, int last, int lds) {
    for (int j = 0; j < KT_CHUNKS * (p.ktiles + 1); j++) {
        const int o = table_entry<REST>(p, j);
        for (const int at : {operand_at<REST>(first, o), operand_at<REST>(last, o)})
            if (at < 0 || at + 16 > lds) return false;
    }
    return true;
}

int main() {
    int l[9];
    while (scanf("%d %d %d %d %d %d %d %d %d", l, l + 1, l + 2, l + 3, l + 4, l + 5, l + 6, l + 7, l + 8) == 9) {
        const int kH = l[5], kW = l[6];
        Params p{};
        int lds = 0;
        if (l[2] + 2 * l[8] < kH || l[3] + 2 * l[8] < kW || !tpl::make_plan(p, &lds, l[0], l[2], l[3], l[1], l[4], kH, kW, l[7], l[8])) {
            printf("none\n");
            continue;
        }
        int most = 0;
        for (int m0 = 0; m0 < p.M; m0 += BLOCK_ROWS) {
            const int last = (m0 + BLOCK_ROWS < p.M ? m0 + BLOCK_ROWS : p.M) - 1, row0 = staged_row(p, m0);
            const int rows = staged_row(p, last) + kH - row0;
            if (rows > most) most = rows;
            // the last staged chunk
            const long long wrote = (long long)(rows - 1) * p.row_bytes + (long long)(p.row_pixels - 1) * p.pixel_bytes + p.group * 16;
            int corner = 0;                         // of the pixel that lies furthest back; the block's first is at 0 or behind
            for (int m = m0; m <= last; m++) {
                const int at = (staged_row(p, m) - row0) * p.row_bytes + m % p.by_OW.d * p.stride * p.pixel_bytes;
                if (at > corner) corner = at;
            }
            const bool inside = tpl::has_rest(p) ? operands_inside<true>(p, p.patch_offset, p.patch_offset + corner, lds)
                                                 : operands_inside<false>(p, p.patch_offset, p.patch_offset + corner, lds);
            if (p.patch_offset + wrote > lds || !inside || p.real_pixels > p.W ||
                p.pad + p.real_pixels > p.row_pixels || (p.real_pixels + p.pad < p.row_pixels && p.real_pixels < p.W)) {
                printf("out of bounds\n");
                return 1;
            }
        }
        const long long rows = tpl::staged_rows(p.OH, p.by_OW.d, kH, p.stride, BLOCK_ROWS < p.M ? BLOCK_ROWS : p.M);
        if (most > rows) return 1;
        printf("%d %lld %d\n", lds, rows * p.row_bytes, p.blocks);
    }
    return 0;
}
