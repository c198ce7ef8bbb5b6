// Line lengths of the general pruned FFT, every sixth of the table (the files
// only divide the compile time).
#include "mn_fftg.h"

namespace mn {

const FgEntry *fg_entries_e(int *count) {
    static const FgEntry table[] = {
        fg::entry<10>(), fg::entry<24>(), fg::entry<40>(), fg::entry<64>(), fg::entry<96>(),
        fg::entry<135>(), fg::entry<192>(), fg::entry<250>(), fg::entry<324>(),
        fg::entry<432>(), fg::entry<540>(), fg::entry<675>(), fg::entry<810>(),
        fg::entry<1024>(), fg::entry<1250>(), fg::entry<1500>(), fg::entry<1875>()};
    *count = (int)(sizeof(table) / sizeof(table[0]));
    return table;
}

}  // namespace mn
