/*
 * grammar_table.h -- the receipt validator (grammar_scan.h) as a transition table
 * over its reachable states, made from the scanner itself at compile time: one
 * lookup per byte in place of a switch that the lanes of a wave take apart.
 */
#ifndef DLK_GRAMMAR_TABLE_H
#define DLK_GRAMMAR_TABLE_H

#include "grammar_scan.h"

namespace dlk {

constexpr int kReceiptStates = 96;           /* reachable, the rejecting state 0 among them */
constexpr int kReceiptClasses = 32;          /* bytes that no state tells apart share a class */
constexpr int kReceiptKeys = 14 * 16 * 2 * 2;

struct ReceiptTable {
    int states;
    uint8_t cls[256];
    uint8_t next[kReceiptStates][kReceiptClasses];
    uint8_t id[kReceiptKeys];                /* of the state with this key; 0: none */
};

/* All that a receipt state is, for states the scanner can be in (-1: it cannot):
 * of the previous byte only whether it was a backslash matters. */
DLK_GHD int dlk_receipt_key(const dlk_scan_state *s) {
    if (s->mode != DLK_GRAMMAR_RECEIPT || s->pc < 0 || s->pc > DLK_RC_WS6 || s->n < 0 || s->n > 15 || s->flag > 1)
        return -1;
    return ((s->pc * 16 + s->n) * 2 + s->flag) * 2 + (s->prev == '\\' ? 1 : 0);
}

constexpr ReceiptTable make_receipt_table() {
    ReceiptTable t{};
    /* a class of its own for each byte that is compared with, one each for the
     * other spaces and digits, 0 for the rest */
    const char alone[] = "{}[],:\"\\_2bdoxtecn";
    int classes = 1;
    uint8_t of[kReceiptClasses] = {};        /* a byte of each class */
    for (int i = 0; alone[i]; i++) {
        of[classes] = (uint8_t)alone[i];
        t.cls[(uint8_t)alone[i]] = (uint8_t)classes++;
    }
    of[classes] = ' ';
    for (int c = 0; c < 256; c++)
        if (dlk_isspace((uint8_t)c)) t.cls[c] = (uint8_t)classes;
    classes++;
    of[classes] = '0';
    for (int c = 0; c < 256; c++)
        if (dlk_isdigit((uint8_t)c) && t.cls[c] == 0) t.cls[c] = (uint8_t)classes;
    classes++;
    dlk_scan_state seen[kReceiptStates] = {};
    dlk_scan_init(&seen[1], DLK_GRAMMAR_RECEIPT);
    t.states = 2;
    t.id[dlk_receipt_key(&seen[1])] = 1;
    for (int s = 1; s < t.states; s++)
        for (int c = 0; c < classes; c++) {
            dlk_scan_state x = seen[s];
            dlk_scan_step(&x, of[c]);
            if (!dlk_scan_ok(&x)) continue;
            const int key = dlk_receipt_key(&x);
            if (t.id[key] == 0) {
                t.id[key] = (uint8_t)t.states;
                seen[t.states++] = x;
            }
            t.next[s][c] = t.id[key];
        }
    return t;
}

#if defined(__HIPCC__)
__device__ const ReceiptTable kReceiptTable = make_receipt_table();
#endif

}  // namespace dlk

#endif
