/*
 * Host view of a finalized BSIM4 instance set, for the code that lays its
 * tables out on the device: the set itself (ngmi_bsim4_eval) and the batched
 * transient.
 */
#ifndef NGMI_SET_TABLE_H
#define NGMI_SET_TABLE_H

#include <vector>
#include "ngmi_internal.h"

namespace ngmi {

/* complete field rows ([records][B4F__COUNT]) and each instance's record;
 * nc = the per-instance columns in use (see bsim4_dev.h).  ok = false: the
 * instances share too few records, and the column form is used. */
struct SetRecords {
    bool ok = false;
    int nc = 0;
    std::vector<double> rec;
    std::vector<int> rec_of;
};

const B4Tab *set_table(const ngmi_bsim4_set *s);
const SetRecords *set_records(const ngmi_bsim4_set *s);
/* ngmi_bsim4_set_finalize without the device tables */
int set_finalize_host(ngmi_bsim4_set *s);
/* the column form's device tables */
int set_upload_columns(ngmi_bsim4_set *s);
/* all B4_NC_GEOM instance columns, in tiles ([tile][column][64]), of the
 * storage order at[] (instance, or -1: a hole) */
void set_tiles(const ngmi_bsim4_set *s, const std::vector<int> &at, std::vector<double> &tiles);

}  // namespace ngmi

#endif
