// Line lengths of the general pruned FFT, every sixth of the table (the files
// only divide the compile time).
#include "mn_fftg.h"

namespace mn {

const FgEntry *fg_entries_c(int *count) {
    static const FgEntry table[] = {
        fg::entry<8>(), fg::entry<18>(), fg::entry<32>(), fg::entry<54>(), fg::entry<81>(),
        fg::entry<125>(), fg::entry<162>(), fg::entry<240>(), fg::entry<300>(),
        fg::entry<400>(), fg::entry<500>(), fg::entry<640>(), fg::entry<768>(),
        fg::entry<972>(), fg::entry<1200>(), fg::entry<1440>(), fg::entry<1728>(),
        fg::entry<2025>()};
    *count = (int)(sizeof(table) / sizeof(table[0]));
    return table;
}

}  // namespace mn
