// Line lengths of the general pruned FFT, every sixth of the table (the files
// only divide the compile time).
#include "mn_fftg.h"

namespace mn {

const FgEntry *fg_entries_f(int *count) {
    static const FgEntry table[] = {
        fg::entry<12>(), fg::entry<25>(), fg::entry<45>(), fg::entry<72>(), fg::entry<100>(),
        fg::entry<144>(), fg::entry<200>(), fg::entry<256>(), fg::entry<360>(),
        fg::entry<450>(), fg::entry<576>(), fg::entry<720>(), fg::entry<864>(),
        fg::entry<1080>(), fg::entry<1280>(), fg::entry<1536>(), fg::entry<1920>()};
    *count = (int)(sizeof(table) / sizeof(table[0]));
    return table;
}

}  // namespace mn
