// Host side of FP32 gemm_ring.hip, one configuration of it: exits with 1 unless the offset that reads zeros is a whole 16-byte piece
// behind the buffer of every K tile of every operand that gemm() takes, the largest ones of 4 GiB among them.
#include "gemm_ring.hip"

int main() {
    const unsigned beyond = (unsigned)OOB_OFFSET;
    unsigned long long most = 0;
    for (long long K = 1; K < 0x7fffffffLL; K = K * 5 / 4 + 1) {
        const long long last = 0x100000000LL / (4 * K) / 4 * 4;          // the first ld that is too much, or near it
        for (long long ld = last > 64 ? last - 64 : 4; ld <= last + 64 && ld <= 0x7ffffffcLL; ld += 4) {
            if (!tpl::operand_fits((int)K, (int)ld)) continue;
            const unsigned long long bytes = (unsigned long long)K * ld * 4;
            if (bytes > most) most = bytes;
            for (const int rows : {(int)K, (int)(K < 2 * BK ? K : 2 * BK), (int)(K % BK ? K % BK : BK)})
                if (tile_bytes(rows, (int)ld, 0) > beyond) {
                    printf("%lld rows of %lld floats: zeros are read at byte %u of %u\n", K, ld, beyond, tile_bytes(rows, (int)ld, 0));
                    return 1;
                }
        }
    }
    if (most < 0xfff00000ULL || beyond % 16 != 0) {
        printf("%u, operands up to %llu\n", beyond, most);
        return 1;
    }
    return 0;
}
