// Bounds of the plans whose entities' first pairs are exported (pg_plan_entity_pairs):
// those of the table assembly by rows (k_table_rows, small p = 2 and 3 systems), whose
// workgroup keeps an entity's rows, pairs and elements in LDS.  The other assembly
// (pg_rows.hip) takes entities of any size and finds the first pairs by bisection
// where they are not given.
#pragma once

namespace pg {

constexpr int kRowAsmMaxLen = 192;  // columns of an entity's rows
constexpr int kRowAsmMaxInc = 24;   // elements containing one entity
constexpr int kRowAsmMaxPairs = 96;  // entities coupled to one entity

}  // namespace pg
