// Chip-resident time loop, FDORDER 12, acoustic, VTI, TTI and SH.
#define DN_F 6
#define DN_GROUP 1
#include "dn_resident_inst.inc"
