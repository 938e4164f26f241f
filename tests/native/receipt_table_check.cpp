/* The receipt validator's transition table (hip/grammar_table.h) against the scanner that it is made from, over every
 * reachable state, every byte, and random strings.  Prints "<states> <checked> <mismatches>".  Test infrastructure. */
#include <stdio.h>
#include <stdlib.h>

#include "../../diskllm_amd/csrc/hip/grammar_table.h"

static constexpr dlk::ReceiptTable T = dlk::make_receipt_table();

int main() {
    long checked = 0, bad = 0;
    const char *pieces[] = {"{", "\"bbox_2d\":", "\"bbox_2d\"", " ", "\t\n", "[", "1", "20", ",", ", ", "]", "}", "\"text_content\":",
                            "\"", "\\", "ab", "\\\"", "x", "\x80", "2d", "n", "e"};
    srand(7);
    for (int it = 0; it < 400000; it++) {
        dlk_scan_state s;
        dlk_scan_init(&s, DLK_GRAMMAR_RECEIPT);
        int id = 1;
        const char *lead = "{\"bbox_2d\":[1,2,3,4],\"text_content\":\"a\"}";
        for (int n = rand() % 44; n > 0 && *lead; n--, lead++) {
            dlk_scan_step(&s, (uint8_t)*lead);
            id = T.next[id][T.cls[(uint8_t)*lead]];
        }
        for (int piece = 0; piece < 6; piece++) {
            const char *p = pieces[rand() % (sizeof pieces / sizeof *pieces)];
            char any[2] = {(char)(rand() % 255 + 1), 0};
            if (rand() % 4 == 0) p = any;
            for (; *p; p++) {
                dlk_scan_step(&s, (uint8_t)*p);
                id = T.next[id][T.cls[(uint8_t)*p]];
                const int want = dlk_scan_ok(&s) ? T.id[dlk::dlk_receipt_key(&s)] : 0;
                checked++;
                if (id != want || (dlk_scan_ok(&s) && want == 0)) bad++;
            }
        }
    }
    printf("%d %ld %ld\n", T.states, checked, bad);
    return bad != 0;
}
